"""Small linears on their own kernel (device storage) against the CPU oracle:
one and several 16-row groups, both block widths, k of one vector, of whole and
ragged 128-byte lines, of several runs per wave and of no whole vectors, output
counts that are no multiple of 16. Bounds as in test_gpu_linear.py."""
import numpy as np
import pytest

from tests.test_gpu_linear import abs_weight, check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("rows,inner,out", [
    (5, 8, 1), (16, 64, 16), (17, 72, 33), (33, 1000, 130), (64, 2048, 100), (7, 4096, 50),
    (20, 3080, 4100), (64, 264, 4112), (31, 136, 2500), (5, 1416, 1536), (50, 520, 1300),
    # rows at any element's alignment, cut vectors; one to four input rows
    (1, 9, 7), (4, 37, 40), (2, 291, 100), (40, 75, 90), (17, 1003, 70), (33, 131, 4099),
    # 64 rows per block
    (65, 8, 17), (130, 1500, 500), (200, 261, 140), (260, 120, 1030), (1000, 77, 33),
])
def test_few_rows(sdk, orc, dtype, with_bias, rows, inner, out):
    x = orc.normal((rows, inner), 81, 0, 0.0, 1.0, dtype)
    w = orc.normal((out, inner), 81, 1, 0.0, 0.1, dtype)
    b = orc.normal((out,), 81, 2, 0.0, 1.0, dtype) if with_bias else None
    y = sdk.tensor(dtype, (rows, out))
    sdk.call(f"tensor_linear_{dtype}", sdk.from_numpy(x), sdk.from_numpy(w),
             None if b is None else sdk.from_numpy(b), y)
    check(y.download(), orc.linear(x, w, b), abs_weight(x, w, b), dtype, f"{rows} {inner} {out}")


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("rows,inner,out", [(20, 72, 40), (20, 75, 40), (90, 75, 300)])
def test_special_values_stay_in_their_rows(sdk, dtype, rows, inner, out):
    """An infinite input and a NaN weight reach their own row and column only,
    also in rows whose last line is ragged."""
    x = np.ones((rows, inner), np.float32).astype("f2" if dtype == "f16" else "f4")
    w = np.ones((out, inner), x.dtype)
    x[18, inner - 1] = np.inf
    w[39, 64] = np.nan
    y = sdk.tensor(dtype, (rows, out))
    sdk.call(f"tensor_linear_{dtype}", sdk.from_numpy(x), sdk.from_numpy(w), None, y)
    got = y.download()
    assert np.isnan(got[:, 39]).all() and np.isposinf(got[18, :39]).all()
    assert (np.delete(got, 18, 0)[:, :39] == inner).all()


# either side of the limits on a row's bytes and on the blocks
@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("rows,inner,out", [(100, 3072, 70), (100, 3073, 70), (520, 1536, 40), (520, 1537, 40),
                                            (300, 775, 700), (300, 776, 700), (512, 2048, 500), (700, 800, 1000),
                                            (700, 801, 1000), (520, 640, 200), (64, 1664, 2048), (64, 1700, 2048)])
def test_limits_of_the_small_kernel(sdk, orc, dtype, rows, inner, out):
    test_few_rows(sdk, orc, dtype, True, rows, inner, out)
