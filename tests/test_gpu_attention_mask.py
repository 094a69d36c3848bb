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
