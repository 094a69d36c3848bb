"""Attention of few query rows (decoding, short chunks) against the CPU oracle:
the query heads of a kv head packed into rows, keys in parts over blocks.
Bounds as in test_gpu_attention.py."""
import numpy as np
import pytest

from tests.test_gpu_attention import check, inputs, run_device

pytestmark = pytest.mark.gpu

# batch, q heads, kv heads, q len, kv len, head dim, value dim
DECODE_SHAPES = [
    (1, 1, 1, 1, 1, 64, 64),
    (1, 8, 2, 1, 31, 128, 128),        # one partial tile
    (2, 6, 3, 1, 33, 64, 64),
    (1, 16, 1, 1, 640, 128, 128),      # a full tile of rows
    (1, 17, 1, 1, 300, 64, 64),        # a second row group with one row
    (3, 4, 2, 5, 129, 64, 128),        # values wider than keys
    (1, 12, 4, 3, 2000, 128, 128),     # several parts, ragged last one
    (2, 2, 2, 16, 1500, 64, 64),       # no sharing, 16 positions
    (1, 8, 2, 8, 777, 128, 128),       # 32 rows: two row groups
    (1, 64, 1, 1, 1100, 80, 80),       # 64 rows, padded dims
    (1, 4, 2, 9, 5, 64, 64),           # fewer keys than queries
    (1, 5, 1, 2, 450, 8, 16),
    (1, 3, 3, 1, 900, 40, 24),
    (1, 4, 1, 1, 700, 96, 72),
    (1, 2, 1, 3, 600, 136, 256),
    (1, 10, 5, 1, 1300, 256, 136),
    (130, 1, 1, 1, 1100, 64, 64),      # parts for half a chip of blocks
    (260, 1, 1, 1, 90, 128, 128),      # a block per CU: keys whole
]


@pytest.mark.parametrize("shape", DECODE_SHAPES)
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("causal,masked", [(False, False), (True, False), (False, True), (True, True)])
def test_decode(sdk, orc, shape, dtype, causal, masked):
    q, k, v, mask = inputs(orc, shape, dtype, 75, masked)
    scale = 1.0 / np.sqrt(shape[5])
    got = run_device(sdk, q, k, v, mask, scale, causal, dtype)
    want = orc.sdpa(q, k, v, mask, scale, causal)
    weight = orc.sdpa_abs_weight(q, k, v, mask, scale, causal)
    check(got, want, weight, dtype, f"{shape} causal={causal} mask={masked}")


@pytest.mark.parametrize("dtype,scale", [("f16", -0.2), ("f16", 0.0), ("f16", 3.0), ("f32", -0.2), ("f32", 0.2)])
@pytest.mark.parametrize("direction", [1.0, -1.0])
def test_decode_maxima(sdk, orc, dtype, scale, direction):
    """Scores climbing or falling along the keys (the running maximum moves on
    most tiles, or on the first only), scales of either sign."""
    shape = (1, 8, 2, 2, 1200, 64, 64)
    q, k, v, _ = inputs(orc, shape, dtype, 76, False)
    q[..., 0] = 4.0
    k[..., :, 0] = (direction * 3.0 * np.arange(1200) / 1200).astype(k.dtype)
    got = run_device(sdk, q, k, v, None, scale, False, dtype)
    check(got, orc.sdpa(q, k, v, None, scale, False), orc.sdpa_abs_weight(q, k, v, None, scale, False),
          dtype, f"scale={scale} direction={direction}")


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("dim", [64, 72, 128, 256])
@pytest.mark.parametrize("lk", [70, 1500])
def test_decode_special_rows(sdk, orc, dtype, dim, lk):
    """Per kv head: a NaN key (every row that sees a key is NaN, also when
    its only visible key is in a later tile; a row that sees nothing is
    zero), an infinite value (its column is infinite), a row seeing nothing."""
    shape = (1, 4, 2, 6, lk, dim, dim)
    q, k, v, mask = inputs(orc, shape, dtype, 77, True)
    mask[3, :] = -np.inf
    mask[5, :] = -np.inf
    mask[5, lk - 1] = 0.0
    k[0, 0, 7, dim - 1] = np.nan
    v[0, 1, 9, dim - 1] = np.inf
    got = run_device(sdk, q, k, v, mask, 0.1, False, dtype)
    want = orc.sdpa(q, k, v, mask, 0.1, False)
    assert (got[0, :, 3] == 0).all()
    assert np.isnan(got[0, :2][:, [0, 1, 2, 4, 5]]).all()
    rows = [0, 1, 2, 4]
    assert np.isposinf(got[0, 2:][:, rows, dim - 1]).all()
    tol = 4e-3 if dtype == "f16" else 2e-5
    g = got[0, 2:][:, rows, :dim - 1].astype(np.float64)
    w = want[0, 2:][:, rows, :dim - 1].astype(np.float64)
    assert np.allclose(g, w, rtol=tol, atol=tol)


@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_decode_last_value_infinite(sdk, orc, dtype):
    """An infinite value in the last key, which the loads past the end repeat
    with weight zero."""
    q, k, v, _ = inputs(orc, (1, 2, 1, 1, 45, 64, 64), dtype, 78, False)
    v[0, 0, 44, 3] = -np.inf
    got = run_device(sdk, q, k, v, None, 0.1, False, dtype)
    want = orc.sdpa(q, k, v, None, 0.1, False)
    assert np.isneginf(got[..., 3]).all() and np.isneginf(want[..., 3]).all()
    keep = [i for i in range(64) if i != 3]
    tol = 4e-3 if dtype == "f16" else 2e-5
    assert np.allclose(got[..., keep].astype(np.float64), want[..., keep].astype(np.float64), rtol=tol, atol=tol)


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("shape", [(1, 4, 2, 2, 70, 64, 64), (1, 4, 2, 2, 1500, 128, 128),
                                   (1, 2, 2, 70, 90, 72, 72), (1, 2, 1, 40, 700, 96, 96)])
def test_output_in_place_of_queries(sdk, orc, shape, dtype):
    """out is q: rows that an infinite value reaches are the same as with an
    output of its own (a second pass over such a row must not read a q that the
    first has overwritten)."""
    q, k, v, _ = inputs(orc, shape, dtype, 79, False)
    v[0, 0, shape[4] - 3, 5] = np.inf
    want = orc.sdpa(q, k, v, None, 0.1, False)
    weight = orc.sdpa_abs_weight(q, k, v, None, 0.1, False)
    tq = sdk.from_numpy(q)
    sdk.call(f"tensor_sdpa_device_{dtype}", tq, sdk.from_numpy(k), sdk.from_numpy(v), None, 0.1, 0, tq)
    got = tq.download()
    odd = np.isinf(want)
    assert odd.any() and np.array_equal(got[odd], want[odd])
    check(got[~odd], want[~odd], weight[~odd], dtype, f"{shape} in place")
