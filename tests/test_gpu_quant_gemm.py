"""Quantized linears of many rows (the tiled matrix form and the rule that picks
it) against the oracle's chain, with the bounds of test_gpu_linear.py: one f16
ulp, or 2e-3 of sum |x w| (the f16 reduction bound)."""
import numpy as np
import pytest

from tests.helpers import f16_ulps

pytestmark = pytest.mark.gpu

# rows, in, out: edges of 32-, 64- and 128-row tiles, of 128 columns, of the
# two-block step (an odd number of blocks) and of the 8-XCD grid
SHAPES = [(17, 64, 40), (33, 96, 130), (64, 1056, 257), (65, 32, 1), (100, 992, 777), (129, 160, 1031),
          (300, 2048, 1300), (513, 96, 129), (700, 288, 2049), (1500, 64, 640), (260, 64, 9000)]


@pytest.mark.parametrize("fmt", [1, 2])
@pytest.mark.parametrize("shape", SHAPES)
def test_many_rows(sdk, orc, fmt, shape):
    rows, inner, out = shape
    w = orc.normal((out, inner), 95, 0, 0.0, 0.05)
    ok, packed, message = sdk.quantize(w, fmt)
    assert ok, message
    x = orc.normal((rows, inner), 95, 1, 0.0, 1.0)
    x[rows // 2, inner - 1] = np.inf          # rows redone by the reference's chain
    x[rows - 1, 0] = np.nan
    ty = sdk.tensor("f16", (rows, out))
    sdk.call("tensor_linear_q8_0_f16" if fmt == 1 else "tensor_linear_q4_0_f16", sdk.from_numpy(x),
             sdk.from_numpy(packed.view(np.uint8).reshape(packed.shape), dtype="u8"), ty)
    got = ty.download()
    scale = packed[..., :2].copy().view(np.float16).astype(np.float64)
    if fmt == 1:
        q = packed[..., 2:].view(np.int8).astype(np.float64)
    else:
        body = packed[..., 2:]
        q = np.concatenate([body & 15, body >> 4], axis=-1).astype(np.float64) - 8
    wd = (q * scale).reshape(out, inner)
    finite = np.isfinite(x.astype(np.float32)).all(-1)
    xd = x[finite].astype(np.float64)
    want, weight = xd @ wd.T, np.abs(xd) @ np.abs(wd).T
    g = got[finite]
    # (the exact value rounded once; the oracle's chain is a few f32 roundings away)
    good = (f16_ulps(g, want.astype(np.float16)) <= 1) | (np.abs(g.astype(np.float64) - want) <= 2e-3 * weight)
    assert good.all(), f"{(~good).sum()} of {good.size} off"
    # the infinite and the NaN row: the sign of the weight, NaN for a zero weight
    last = wd[:, inner - 1]
    row = got[rows // 2]
    assert np.isnan(row[last == 0]).all()
    assert np.array_equal(row[last != 0], np.where(last[last != 0] > 0, np.inf, -np.inf).astype(np.float16))
    assert np.isnan(got[rows - 1]).all()
