"""Sum + max and argmax around the sizes where the launch changes: one block,
32 KiB, 128 KiB and 1 MiB chunks, one and several partials per folding lane."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ONE_BLOCK, SMALL, MID = 1024 * 8 * 4, 32768 // 4, 131072 // 4   # floats


@pytest.mark.parametrize("n", [2, 1023, ONE_BLOCK - 1, ONE_BLOCK + 3, ONE_BLOCK + 4, 5 * SMALL + 6,
                               1024 * SMALL, 1024 * SMALL + 4, 1024 * MID, 1024 * MID + 20])
def test_sum_max_sizes(sdk, orc, n):
    x = orc.uniform((n,), 45, 0, -1.0, 1.0)
    tx, ts, tm = sdk.from_numpy(x), sdk.tensor("f64", (1,)), sdk.tensor("f32", (1,))
    for at, value in ((None, 0.0), (0, 2.5), (n // 2, 3.5), (n - 1, 4.5), (n - 1, np.nan)):
        if at is not None:
            x[at] = value
            tx.upload(x)
        sdk.call("tensor_sum_max_f32", tx, ts, tm)
        want_s, abs_s, want_m = orc.sum_max(x)
        if np.isnan(value):
            assert np.isnan(ts.download()[0]) and np.isnan(tm.download()[0])
            continue
        # f32 sums of 32 values, f64 above: 32 roundings of a group's magnitude
        assert abs(float(ts.download()[0]) - want_s) <= 32 * 2.0 ** -24 * abs_s
        assert tm.download()[0] == want_m


@pytest.mark.parametrize("dtype,vec", [("f16", 8), ("f32", 4)])
@pytest.mark.parametrize("n_of", [lambda v: 1, lambda v: v + 1, lambda v: 1024 * 8 * v - 1,
                                  lambda v: 1024 * 8 * v + v - 1, lambda v: 1024 * 8 * v + v])
def test_argmax_sizes(sdk, orc, dtype, vec, n_of):
    n = n_of(vec)
    x = orc.uniform((n,), 46, 0, -1.0, 1.0, dtype)
    tx, ti = sdk.from_numpy(x), sdk.tensor("u32", (1,))
    for at in (0, n // 3, n - 1):
        x[at] = 2.0                      # ties: the first of the maxima wins
        tx.upload(x)
        sdk.call(f"tensor_argmax_{dtype}", tx, ti)
        assert ti.download()[0] == int(np.argmax(x))
        x[at] = 0.0
    x[:] = -np.inf
    tx.upload(x)
    sdk.call(f"tensor_argmax_{dtype}", tx, ti)
    assert ti.download()[0] == 0


@pytest.mark.parametrize("n", [(1 << 26) - 4, (1 << 26) + 3])
def test_sum_max_around_the_largest_chunk(sdk, orc, n):
    """2048 chunks of 128 KiB (two partials per folding lane), 256 of 1 MiB."""
    x = orc.uniform((n,), 47, 0, -1.0, 1.0)
    x[n - 1], x[n // 3] = 2.5, 3.5
    ts, tm = sdk.tensor("f64", (1,)), sdk.tensor("f32", (1,))
    sdk.call("tensor_sum_max_f32", sdk.from_numpy(x), ts, tm)
    want_s, abs_s, want_m = orc.sum_max(x)
    assert abs(float(ts.download()[0]) - want_s) <= 32 * 2.0 ** -24 * abs_s
    assert tm.download()[0] == want_m
