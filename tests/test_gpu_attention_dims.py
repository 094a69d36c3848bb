"""Attention at head dims other than 64 and 128 against the CPU oracle.

Rows of up to 256 elements that are whole 16-byte vectors run on the flash
kernels compiled for padded dims; the bounds are those of
test_gpu_attention.py (f16 P is carried as an f16 pair there, so nothing is
allowed for its rounding beyond them)."""
import numpy as np
import pytest

from tests.test_gpu_attention import check, inputs, run_device

pytestmark = pytest.mark.gpu

# batch, q heads, kv heads, q len, kv len, head dim, value dim
DIM_SHAPES = [
    (1, 2, 1, 33, 65, 8, 8),        # one vector per f16 row
    (1, 2, 2, 40, 70, 32, 24),      # narrower values
    (1, 4, 2, 65, 130, 40, 48),     # padded to 80
    (2, 3, 3, 100, 90, 72, 72),
    (1, 16, 4, 257, 200, 80, 80),   # 128-query blocks
    (1, 2, 1, 70, 700, 88, 96),     # key range split, wider values
    (1, 70, 70, 130, 70, 96, 96),   # one round of 128-query blocks
    (1, 72, 8, 520, 66, 80, 72),    # 256-query blocks (f16)
    (1, 2, 2, 30, 520, 112, 120),
    (1, 2, 2, 66, 300, 136, 256),   # 256-wide tiles
    (1, 33, 33, 130, 70, 256, 144),
    (1, 2, 1, 1, 777, 80, 80),      # one query, split
]


@pytest.mark.parametrize("shape", DIM_SHAPES)
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("causal,masked", [(False, False), (True, False), (True, True)])
def test_padded_head_dims(sdk, orc, shape, dtype, causal, masked):
    q, k, v, mask = inputs(orc, shape, dtype, 71, masked)
    scale = 1.0 / np.sqrt(shape[5])
    got = run_device(sdk, q, k, v, mask, scale, causal, dtype)
    want = orc.sdpa(q, k, v, mask, scale, causal)
    weight = orc.sdpa_abs_weight(q, k, v, mask, scale, causal)
    check(got, want, weight, dtype, f"{shape} causal={causal} mask={masked}")


@pytest.mark.parametrize("dims", [(12, 4), (36, 68), (100, 132)])
def test_f32_rows_of_whole_vectors(sdk, orc, dims):
    """f32 rows of 4 mod 8 elements (the merge's last group holds 4)."""
    for shape in [(1, 2, 1, 40, 50) + dims, (1, 1, 1, 8, 900) + dims]:
        q, k, v, _ = inputs(orc, shape, "f32", 72, False)
        got = run_device(sdk, q, k, v, None, 0.1, False, "f32")
        check(got, orc.sdpa(q, k, v, None, 0.1, False),
              orc.sdpa_abs_weight(q, k, v, None, 0.1, False), "f32", str(shape))


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("dim", [72, 96, 200])
@pytest.mark.parametrize("lk", [70, 600])
def test_special_rows(sdk, orc, dtype, dim, lk):
    """Rows wholly masked, a NaN key and an infinite value, against the oracle.
    Head 0 holds the NaN key: every row is NaN (row 5 through a key in a later
    tile than its only visible one), except row 3, which sees nothing and is
    zero. Head 1 holds the infinite value: its column is infinite in every row
    but 3 and 5, whose weight for that key is 0 (0 * inf is not compared)."""
    shape = (1, 2, 2, 40, lk, dim, dim)
    q, k, v, mask = inputs(orc, shape, dtype, 73, True)
    mask[3, :] = -np.inf
    mask[5, :] = -np.inf
    mask[5, lk - 1] = 0.0
    k[0, 0, 7, dim - 1] = np.nan
    v[0, 1, 9, dim - 1] = np.inf
    got = run_device(sdk, q, k, v, mask, 0.1, False, dtype)
    want = orc.sdpa(q, k, v, mask, 0.1, False)
    assert (got[0, 0, 3] == 0).all() and (got[0, 1, 3] == 0).all()
    rows = [i for i in range(40) if i != 3]
    assert np.isnan(got[0, 0, rows]).all()
    rows.remove(5)
    assert np.isposinf(got[0, 1, rows, dim - 1]).all() and np.isposinf(want[0, 1, rows, dim - 1]).all()
    tol = 4e-3 if dtype == "f16" else 2e-5
    g, w = got[0, 1, rows, :dim - 1].astype(np.float64), want[0, 1, rows, :dim - 1].astype(np.float64)
    assert np.allclose(g, w, rtol=tol, atol=tol)


@pytest.mark.parametrize("dim", [64, 72, 128])
def test_f32_nan_before_the_visible_key(sdk, orc, dim):
    """A NaN score in a tile where the row sees nothing yet makes the whole
    row NaN, in both halves of the wave."""
    q, k, v, mask = inputs(orc, (1, 1, 1, 8, 70, dim, dim), "f32", 74, True)
    mask[5, :] = -np.inf
    mask[5, 69] = 0.0
    k[0, 0, 7, 0] = np.nan
    got = run_device(sdk, q, k, v, mask, 0.1, False, "f32")
    assert np.isnan(got[0, 0, 5]).all()


@pytest.mark.parametrize("dim", [40, 72, 80, 88, 96, 136, 248])
def test_merged_rows_are_done_again_whole(sdk, orc, dim):
    """Keys cut into parts, an infinite value that every row sees: the merge
    does those rows again, each as a whole (a row of 9 to 12 groups of 8 once
    lay in two waves, and the one that had nothing to do again stored its own
    columns at any time). An output in place of the queries takes the row
    kernel, whose outputs every column must equal, each time."""
    q, k, v, _ = inputs(orc, (1, 2, 2, 40, 2000, dim, dim), "f16", 75, False)
    v[0, :, 1000, dim - 1] = np.inf
    tq, tk, tv = sdk.from_numpy(q), sdk.from_numpy(k), sdk.from_numpy(v)
    sdk.call("tensor_sdpa_device_f16", tq, tk, tv, None, 0.1, 0, tq)
    rows = tq.download()
    assert np.isposinf(rows[..., dim - 1]).all()
    for _ in range(4):
        got = run_device(sdk, q, k, v, None, 0.1, False, "f16")
        assert np.array_equal(got.view(np.uint16), rows.view(np.uint16))


def test_more_heads_than_a_flash_launch_holds(sdk):
    """2^23 heads of one query and one key: the output is the value row."""
    shape = (1 << 20, 8, 1, 8)
    v = (np.arange(1 << 26, dtype=np.uint32) % 2039).astype(np.float16).reshape(shape)
    tq = tk = sdk.from_numpy(np.ones(shape, np.float16))
    out = sdk.tensor("f16", shape)
    sdk.call("tensor_sdpa_device_f16", tq, tk, sdk.from_numpy(v), None, 0.1, 0, out)
    assert np.array_equal(out.download(), v)
