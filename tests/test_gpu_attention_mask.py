"""Masked attention against the CPU oracle: the flash kernels read the mask as
16-byte vectors at any element alignment, and a ragged last key tile element
by element. Bounds as in test_gpu_attention.py."""
import numpy as np
import pytest

from tests.test_gpu_attention import check, inputs, run_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("dim", [64, 72, 128])
@pytest.mark.parametrize("lq,lk", [(66, 63), (70, 64), (66, 65), (97, 129), (65, 191), (130, 520)])
@pytest.mark.parametrize("causal", [False, True])
def test_masks_of_any_row_length(sdk, orc, dtype, dim, lq, lk, causal):
    """Rows with hidden keys, with the type's lowest value throughout, and
    wholly hidden (zero rows), at odd and even row lengths."""
    shape = (1, 2, 1, lq, lk, dim, dim)
    q, k, v, mask = inputs(orc, shape, dtype, 91, True)
    mask[0, :] = -np.inf
    mask[7, ::3] = -np.inf
    mask[lq - 1, : lk - 1] = -np.inf
    mask[9, :] = np.finfo(mask.dtype).min
    scale = 1.0 / np.sqrt(dim)
    got = run_device(sdk, q, k, v, mask, scale, causal, dtype)
    want = orc.sdpa(q, k, v, mask, scale, causal)
    assert (got[0, :, 0] == 0).all()
    weight = orc.sdpa_abs_weight(q, k, v, mask, scale, causal)
    # row 9: scores rounded to the lowest value's steps are compared for
    # finiteness only
    assert np.isfinite(got).all()
    rows = [i for i in range(lq) if i != 9]
    check(got[:, :, rows], want[:, :, rows], weight[:, :, rows], dtype, f"{dim} {lq} {lk} {causal}")


# batch, q heads, kv heads, q len, kv len, head dim: few rows packed (whole and
# in parts), key tiles whole and in parts
@pytest.mark.parametrize("shape", [(8, 8, 2, 4, 300, 64), (4, 8, 2, 4, 2000, 128), (4, 8, 2, 4, 600, 72),
                                   (4, 8, 2, 4, 2000, 200), (1, 4, 2, 130, 600, 72), (1, 4, 4, 70, 2000, 96),
                                   (2, 4, 2, 150, 700, 200)])
def test_rows_of_the_lowest_value(sdk, orc, shape):
    """f16 rows whose keys all carry the type's lowest value. In f32 such a
    score, about -65504, is rounded to steps of 2^-8: errors uniform within
    2^-9, so the weights are 2^-9 / sqrt(3) off, and the outputs (sums of
    values of mean zero) as much, beside their own rounding, at most
    2^-11 / sqrt(3). A tenth over that; twice the step (scores times log2 e,
    past 65536) gives 1.56e-3."""
    b, h, kh, lq, lk, dim = shape
    q, k, v, _ = inputs(orc, (b, h, kh, lq, lk, dim, dim), "f16", 92, False)
    mask = np.full((lq, lk), np.finfo(np.float16).min, np.float16)
    scale = 1.0 / np.sqrt(dim)
    got = run_device(sdk, q, k, v, mask, scale, False, "f16").astype(np.float64)
    k64, v64 = (np.repeat(a.astype(np.float64), h // kh, axis=1) for a in (k, v))
    s = np.matmul(q.astype(np.float64), k64.transpose(0, 1, 3, 2)) * np.float64(np.float32(scale))
    p = np.exp(s - s.max(-1, keepdims=True))     # (the same mask everywhere)
    want = np.matmul(p / p.sum(-1, keepdims=True), v64)
    error = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert error <= 1.1 * np.hypot(2.0 ** -9, 2.0 ** -11) / np.sqrt(3.0), error
