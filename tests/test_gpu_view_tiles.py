"""Transposing views at the edges of their tiles, with and without operands,
against numpy (one or two IEEE operations in f32, rounded once: exact)."""
import numpy as np
import pytest

from inference_c_amd.sdk import TensorView

pytestmark = pytest.mark.gpu

# stored shape, axis order of the view
CASES = [
    ((64, 64), (1, 0)), ((65, 64), (1, 0)), ((63, 64), (1, 0)), ((67, 129), (1, 0)),
    ((513, 191), (1, 0)), ((300, 66), (1, 0)), ((3, 70, 200), (0, 2, 1)), ((5, 1000, 65), (0, 2, 1)),
    ((40, 900, 1000), (0, 2, 1)),            # four tiles per block (f16)
    ((2, 31, 37, 3), (0, 3, 1, 2)), ((3, 64, 64, 4), (0, 3, 1, 2)), ((1, 50, 41, 2), (0, 3, 1, 2)),
    ((2, 3, 31, 37), (0, 2, 3, 1)), ((1, 16, 65, 9), (0, 2, 3, 1)), ((2, 63, 20, 70), (0, 2, 3, 1)),
    ((33, 17, 65), (2, 0, 1)), ((9, 8, 7, 6), (3, 2, 1, 0)), ((70, 5, 66), (2, 1, 0)),
    ((2, 5000), (1, 0)), ((5000, 2), (1, 0)), ((1, 3), (1, 0)),
]


def broadcast(kind, shape):
    if kind is None:
        return None
    keep = {"last": {len(shape) - 1}, "first": {0}, "second": {1}, "full": set(range(len(shape))),
            "one": set()}[kind]
    return tuple(n if i in keep else 1 for i, n in enumerate(shape))


@pytest.mark.parametrize("shape,order", CASES)
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("add,mul", [(None, None), ("last", None), (None, "last"), ("second", "second"),
                                     ("full", "one"), ("one", "full"), ("last", "first")])
def test_transposing_view(sdk, orc, shape, order, dtype, add, mul):
    np_type = np.float16 if dtype == "f16" else np.float32
    x = orc.normal(shape, 91, 0, 0.0, 1.0, dtype)
    out = tuple(shape[i] for i in order)
    a_shape, m_shape = broadcast(add, out), broadcast(mul, out)
    a = None if add is None else orc.normal(a_shape, 91, 1, 0.0, 1.0, dtype)
    m = None if mul is None else orc.normal(m_shape, 91, 2, 1.0, 1.0, dtype)
    strides = [int(np.prod(shape[i + 1:])) for i in range(len(shape))]
    view = TensorView.make(out, [strides[i] for i in order])
    ty = sdk.tensor(dtype, out)
    sdk.call(f"tensor_view_add_mul_{dtype}", sdk.from_numpy(x), view,
             None if a is None else sdk.from_numpy(a), None if m is None else sdk.from_numpy(m), ty)
    want = np.ascontiguousarray(x.transpose(order)).astype(np.float32)
    if a is not None:
        want = want + a.astype(np.float32)
    if m is not None:
        want = want * m.astype(np.float32)
    assert np.array_equal(ty.download(), want.astype(np_type))


@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_slices_and_gaps(sdk, orc, dtype):
    """An offset and row strides that are not whole vectors; a broadcast
    (stride 0) batch dimension."""
    x = orc.normal((90 * 131 + 7,), 92, 0, 0.0, 1.0, dtype)
    tx = sdk.from_numpy(x)
    for shape, strides, offset in [((77, 80), (1, 131), 7), ((66, 3, 88), (1, 5, 131), 3),
                                   ((4, 70, 65), (0, 1, 100), 1), ((3, 66, 70), (1, 131, 17), 5)]:
        idx = offset + sum(np.arange(n).reshape([-1 if i == d else 1 for i in range(len(shape))]) * s
                           for d, (n, s) in enumerate(zip(shape, strides)))
        ty = sdk.tensor(dtype, shape)
        sdk.call(f"tensor_view_add_mul_{dtype}", tx, TensorView.make(shape, strides, offset), None, None, ty)
        assert np.array_equal(ty.download(), x[idx])


@pytest.mark.parametrize("shape", [(128, 192), (65, 64), (67, 129), (130, 4099), (3000, 1000)])
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("add,mul", [(True, False), (False, True), (True, True)])
def test_output_is_an_operand(sdk, orc, shape, dtype, add, mul):
    """y = view(x) + y, view(x) * y, (view(x) + y) * y: each element of y
    enters once, as it was before the call."""
    np_type = np.float16 if dtype == "f16" else np.float32
    x = orc.normal(shape, 93, 0, 0.0, 1.0, dtype)
    y = orc.normal(shape[::-1], 93, 1, 0.0, 1.0, dtype)
    ty = sdk.from_numpy(y)
    sdk.call(f"tensor_view_add_mul_{dtype}", sdk.from_numpy(x), TensorView.make(shape[::-1], (1, shape[1])),
             ty if add else None, ty if mul else None, ty)
    want = x.T.astype(np.float32)
    if add:
        want = want + y.astype(np.float32)
    if mul:
        want = want * y.astype(np.float32)
    assert np.array_equal(ty.download(), want.astype(np_type))


# many small transposes (more than 4 M elements: large tiles where they fill):
# one element per lane, whole vectors in part of a tile, small and large tiles
@pytest.mark.parametrize("shape", [(1100000, 2, 2), (700001, 2, 3), (130000, 5, 7), (65537, 8, 8), (17000, 16, 16),
                                   (11000, 20, 20), (7400, 24, 24), (4100, 31, 33), (4200, 32, 32),
                                   (3900, 33, 33), (2700, 40, 40), (2200, 4, 500), (2200, 500, 4), (1100, 504, 8),
                                   (1100, 8, 504), (300, 24, 1000), (300, 1000, 24), (70, 1000, 63)])
@pytest.mark.parametrize("dtype", ["f16", "f32"])
@pytest.mark.parametrize("add,mul", [(None, None), ("full", "second"), (None, "last")])
def test_batched_small_transposes(sdk, orc, shape, dtype, add, mul):
    test_transposing_view(sdk, orc, shape, (0, 2, 1), dtype, add, mul)
