"""Row operations at widths and alignments outside the vector register
kernels' (narrow rows, rows that are not whole 16-byte vectors, long rows of
one block, rows cut over several blocks), against the CPU oracle.

Bounds: f16 one ulp of the oracle's rounding (the f32 value before it differs
by a few f32 roundings, so at most a tie moves); f32 reductions 1e-5 of the
result, as the other reductions here."""
import numpy as np
import pytest

from tests.helpers import assert_f16_ulps, assert_f32_rel

pytestmark = pytest.mark.gpu

# rows, width: edges of 8, 16, 32, 64 lanes, of 2 and 4 waves, of the 1024-lane
# block and of the parts, for f16 (8 per vector) and f32 (4 per vector)
SHAPES = [(1, 8), (3, 9), (37, 32), (70, 63), (5, 64), (33, 65), (9, 127), (40, 129), (17, 255),
          (6, 257), (5, 509), (300, 513), (3, 1001), (2, 2049), (2, 4099), (3, 8195), (3, 16381),
          (130, 16391), (130, 8197), (2, 16391), (1, 32761), (2, 65531), (1, 131069)]


@pytest.mark.parametrize("rows,width", SHAPES)
@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_norms(sdk, orc, rows, width, dtype):
    x = orc.normal((rows, width), 81, 0, 0.3, 1.0, dtype)
    w = orc.uniform((width,), 81, 1, 0.5, 1.5, dtype)
    b = orc.uniform((width,), 81, 2, -0.5, 0.5, dtype)
    tx, tw, tb = (sdk.from_numpy(a) for a in (x, w, b))
    ty = sdk.tensor(dtype, x.shape)

    def same(want, what):
        if dtype == "f16":
            assert_f16_ulps(ty.download(), want, 1, what)
        else:
            assert_f32_rel(ty.download(), want, 1e-5, what)

    def layer(scale, bias):   # closed form in float64
        d = x.astype(np.float64)
        d = d - d.mean(-1, keepdims=True)
        v = d / np.sqrt((d * d).mean(-1, keepdims=True) + 1e-5)
        v = v * scale if scale is not None else v
        return v + bias if bias is not None else v

    sdk.call(f"tensor_rms_norm_{dtype}", tx, tw, 1e-6, ty)
    if dtype == "f16":
        same(orc.rms_norm(x, w, 1e-6), "rms")
    else:   # in float64: the oracle's sequential f32 sum of 131069 squares is itself 1.2e-5 off
        d = x.astype(np.float64)
        same(d / np.sqrt((d * d).mean(-1, keepdims=True) + 1e-6) * w, "rms")
    # a cancelling bias leaves the sum's own rounding: bound by the row's size
    for scale, bias in ((tw, tb), (None, None), (tw, None), (None, tb)):
        sdk.call(f"tensor_layer_norm_{dtype}", tx, scale, bias, 1e-5, ty)
        want = layer(w.astype(np.float64) if scale else None, b.astype(np.float64) if bias else None)
        tol = 2.0 ** -10 if dtype == "f16" else 1e-5
        got = ty.download().astype(np.float64)
        assert (np.abs(got - want) <= tol * np.maximum(np.abs(want), 1.0)).all(), (rows, width)


@pytest.mark.parametrize("rows,width", SHAPES)
@pytest.mark.parametrize("in_place", [False, True])
def test_residual_rms(sdk, orc, rows, width, in_place):
    """Also with the sum written over the input (each element is read before
    any of the row is written)."""
    x = orc.normal((rows, width), 82, 0, 0.0, 1.0)
    r = orc.normal((rows, width), 82, 1, 0.0, 1.0)
    w = orc.uniform((width,), 82, 2, 0.5, 1.5, "f16")
    tx, tr, tw = (sdk.from_numpy(a) for a in (x, r, w))
    ts, ty = (tx if in_place else sdk.tensor("f16", x.shape)), sdk.tensor("f16", x.shape)
    sdk.call("tensor_residual_rms_norm_f16", tx, tr, tw, 1e-6, ts, ty)
    s_ref, y_ref = orc.residual_rms_norm(x, r, w, 1e-6)
    assert np.array_equal(ts.download().view(np.uint16), s_ref.view(np.uint16))
    assert_f16_ulps(ty.download(), y_ref, 1, "residual rms")


def softmax64(x, causal, q_len):
    """The documented rules in float64."""
    s = x.astype(np.float64).copy()
    rows, width = s.shape
    if causal:
        for r in range(rows):
            s[r, (r % q_len) + max(width - q_len, 0) + 1:] = -np.inf
    out = np.zeros_like(s)
    for r in range(rows):
        m = np.fmax.reduce(s[r])
        if m == -np.inf:
            continue
        if m == np.inf:
            hit = s[r] == np.inf
            out[r, hit] = 1.0 / hit.sum()
            continue
        p = np.exp(s[r] - m)
        out[r] = p / p.sum()
    return out


@pytest.mark.parametrize("rows,width", SHAPES)
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("causal", [False, True])
def test_softmax(sdk, orc, rows, width, dtype, causal):
    x = orc.normal((rows, width), 83, 0, 0.0, 2.0, dtype)
    if rows >= 3:   # one row each: a NaN, nothing visible, two +inf keys
        x[0, width - 1 if not causal else 0] = np.nan
        x[1, :] = -np.inf
        x[2, 0] = x[2, width // 2 if not causal else 0] = np.inf
    tx, ty = sdk.from_numpy(x), sdk.tensor(dtype, x.shape)
    sdk.call(f"tensor_softmax_{dtype}", tx, int(causal), ty)
    got = ty.download().astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = softmax64(x, causal, rows)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    # f16: half an ulp (2^-25 absolute among its subnormals); f32: exp and the
    # sum's roundings
    tol = 2.0 ** -10 * want + 2.0 ** -24 if dtype == "f16" else 1e-5 * want + 1e-30
    ok = np.isnan(want) | (np.abs(got - want) <= tol)
    assert ok.all(), f"{(~ok).sum()} of {ok.size} off"


@pytest.mark.parametrize("rows,width", SHAPES)
@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_sum_and_max(sdk, orc, rows, width, dtype):
    x = orc.normal((rows, width), 84, 0, 0.1, 1.0, dtype)
    if rows >= 3:
        x[0, width - 1] = np.nan
        x[1, :] = np.finfo(np.float16 if dtype == "f16" else np.float32).min
        x[2, 0] = -np.inf
    tx, ty = sdk.from_numpy(x), sdk.tensor("f32", (rows,))
    sdk.call(f"tensor_row_max_{dtype}", tx, ty)
    assert np.array_equal(ty.download(), x.max(-1).astype(np.float32), equal_nan=True)
    if rows >= 3:
        x[:3] = 0.5
        tx = sdk.from_numpy(x)
    sdk.call(f"tensor_row_sum_{dtype}", tx, ty)
    # bound by the sum of magnitudes: the rounding of any order of f32 adds
    weight = np.abs(x.astype(np.float64)).sum(-1)
    assert (np.abs(ty.download() - x.astype(np.float64).sum(-1)) <= 1e-5 * weight).all()


def test_softmax_in_place_cut_rows(sdk, orc):
    """y over x, rows cut into parts whose last vector overlaps the one before."""
    for width in (65531, 2047 * 4 * 9 + 1):
        x = orc.normal((2, width), 85, 0, 0.0, 2.0, "f32")
        tx = sdk.from_numpy(x)
        sdk.call("tensor_softmax_f32", tx, 0, tx)
        want = softmax64(x, False, 2)
        assert (np.abs(tx.download() - want) <= 1e-5 * want).all()


# rows cut into parts: whole last vectors, ragged ones that overlap the one
# before, a last part that joined the one before it
@pytest.mark.parametrize("rows,width", [(2, 65536), (3, 65531), (2, 2047 * 8 * 5 + 1)])
@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_cut_rows_in_place(sdk, orc, rows, width, dtype):
    """y over x: every load of a part comes before any store of it."""
    x = orc.normal((rows, width), 87, 0, 0.3, 1.0, dtype)
    w = orc.uniform((width,), 87, 1, 0.5, 1.5, dtype)
    b = orc.uniform((width,), 87, 2, -0.5, 0.5, dtype)
    tw, tb = sdk.from_numpy(w), sdk.from_numpy(b)
    d = x.astype(np.float64)
    c = d - d.mean(-1, keepdims=True)
    soft = softmax64(x, False, rows)
    for name, args, want in (
            ("rms_norm", (tw, 1e-6), d / np.sqrt((d * d).mean(-1, keepdims=True) + 1e-6) * w),
            ("layer_norm", (tw, tb, 1e-5), c / np.sqrt((c * c).mean(-1, keepdims=True) + 1e-5) * w + b),
            ("softmax", (0,), soft)):
        tx = sdk.from_numpy(x)
        sdk.call(f"tensor_{name}_{dtype}", tx, *args, tx)
        got = tx.download().astype(np.float64)
        # as in the tests above: the output's rounding, the sums' in f32
        tol = 2.0 ** -10 if dtype == "f16" else 1e-5
        floor = (2.0 ** -24 if dtype == "f16" else 1e-30) if name == "softmax" else tol
        assert (np.abs(got - want) <= tol * np.abs(want) + floor).all(), name


@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_captured_long_rows(sdk, orc, dtype):
    """Rows that an eager call cuts, with partial results in scratch memory,
    are recorded as one kernel without; replays give what the eager call does
    up to the sums' order."""
    import ctypes
    hip = sdk.lib
    hip.tensor_device_hip_stream.restype = ctypes.c_void_p
    stream = ctypes.c_void_p(hip.tensor_device_hip_stream())
    x = orc.normal((2, 65531), 88, 0, 0.0, 2.0, dtype)
    tx, ty = sdk.from_numpy(x), sdk.tensor(dtype, x.shape)
    call = (f"tensor_softmax_{dtype}", tx, 0, ty)
    want = softmax64(x, False, 2)
    tol = 2.0 ** -10 * want + 2.0 ** -24 if dtype == "f16" else 1e-5 * want + 1e-30
    graph, exe, nodes = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t()
    sdk.call(*call)
    ty.download()
    assert hip.hipStreamBeginCapture(stream, 2) == 0     # relaxed
    try:
        sdk.call(*call)
    finally:
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0
    assert nodes.value == 1
    assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        ty.upload(np.zeros_like(x))
        assert hip.hipGraphLaunch(exe, stream) == 0
        assert (np.abs(ty.download() - want) <= tol).all()
        sdk.call(*call)          # eager work between the replays
        assert (np.abs(ty.download() - want) <= tol).all()
    assert hip.hipGraphExecDestroy(exe) == 0
    assert hip.hipGraphDestroy(graph) == 0
