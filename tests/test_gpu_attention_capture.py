"""Attention recorded into a graph: the calls whose kernels could take pool
scratch for parts of the key range record one kernel and no scratch, and a
replay gives what the eager call gives."""
import ctypes

import numpy as np
import pytest

from tests.test_gpu_attention import check, inputs

pytestmark = pytest.mark.gpu

RELAXED = 2   # hipStreamCaptureModeRelaxed


# batch, q heads, kv heads, q len, kv len, head dim, value dim: a decode step
# and a prompt at a padded dim; eager, both cut the keys into parts
@pytest.mark.parametrize("shape", [(1, 4, 2, 1, 1500, 80, 80), (1, 2, 1, 70, 700, 96, 96)])
@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_captured_sdpa_takes_no_scratch(sdk, orc, shape, dtype):
    hip = sdk.lib   # (its dependencies' symbols are found through it)
    stream_of = hip.tensor_device_hip_stream
    stream_of.restype = ctypes.c_void_p
    stream = ctypes.c_void_p(stream_of())
    q, k, v, _ = inputs(orc, shape, dtype, 80, False)
    tq, tk, tv = sdk.from_numpy(q), sdk.from_numpy(k), sdk.from_numpy(v)
    out = sdk.tensor(dtype, q.shape[:3] + (v.shape[3],))
    graph, exe, nodes = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t()
    call = (f"tensor_sdpa_device_{dtype}", tq, tk, tv, None, 0.1, 0, out)
    sdk.call(*call)          # code objects are loaded before the capture
    out.download()
    assert hip.hipStreamBeginCapture(stream, RELAXED) == 0
    try:
        sdk.call(*call)
    finally:
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0
    assert nodes.value == 1
    assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
    want = orc.sdpa(q, k, v, None, 0.1, False)
    weight = orc.sdpa_abs_weight(q, k, v, None, 0.1, False)
    for replay in range(3):
        out.upload(np.zeros_like(want))
        assert hip.hipGraphLaunch(exe, stream) == 0
        check(out.download(), want, weight, dtype, f"{shape} replay {replay}")
        sdk.call(*call)      # eager work between the replays
        check(out.download(), want, weight, dtype, f"{shape} eager {replay}")
    assert hip.hipGraphExecDestroy(exe) == 0
    assert hip.hipGraphDestroy(graph) == 0


# the modes of capture: global, of the thread, relaxed
@pytest.mark.parametrize("mode", [0, 1, RELAXED])
# a decode step and a prompt whose key parts take scratch memory
@pytest.mark.parametrize("shape", [(1, 8, 2, 1, 3000, 128, 128), (1, 4, 2, 70, 2000, 64, 64)])
@pytest.mark.parametrize("dtype", ["f16", "f32"])
def test_captured_sdpa_keeps_its_scratch(sdk, orc, shape, dtype, mode):
    """The graph's scratch memory is its own: eager calls between the replays
    and a cleared pool (the compute table's release_cache) leave the replays
    right, and equal to the eager call bit for bit."""
    from tests.test_gpu_vtable import Table
    hip = sdk.lib
    hip.tensor_device_hip_stream.restype = ctypes.c_void_p
    stream = ctypes.c_void_p(hip.tensor_device_hip_stream())
    table = ctypes.cast(hip.tensor_compute_hip_backend(), ctypes.POINTER(Table)).contents
    release = ctypes.CFUNCTYPE(None)(table.release_cache)
    q, k, v, _ = inputs(orc, shape, dtype, 81, False)
    tq, tk, tv = sdk.from_numpy(q), sdk.from_numpy(k), sdk.from_numpy(v)
    out = sdk.tensor(dtype, q.shape[:3] + (v.shape[3],))
    other = [sdk.from_numpy(a[..., ::-1].copy()) for a in (q, k, v)]
    aside = sdk.tensor(dtype, out.shape)
    graph, exe, nodes = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t()
    call = (f"tensor_sdpa_device_{dtype}", tq, tk, tv, None, 0.1, 0, out)
    sdk.call(*call)
    eager = out.download()
    check(eager, orc.sdpa(q, k, v, None, 0.1, False), orc.sdpa_abs_weight(q, k, v, None, 0.1, False), dtype,
          f"{shape} eager")
    assert hip.hipStreamBeginCapture(stream, mode) == 0
    try:
        sdk.call(*call)
    finally:
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0
    assert nodes.value == 2      # the parts and their fold
    assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, ctypes.c_size_t(0)) == 0
    assert hip.hipGraphDestroy(graph) == 0     # the executable keeps the memory
    for _ in range(3):
        release()
        out.upload(np.zeros_like(eager))
        sdk.call(f"tensor_sdpa_device_{dtype}", *other, None, 0.2, 0, aside)
        assert hip.hipGraphLaunch(exe, stream) == 0
        sdk.call(f"tensor_sdpa_device_{dtype}", *other, None, 0.3, 0, aside)
        assert np.array_equal(out.download(), eager)
    sdk.synchronize()
    assert hip.hipGraphExecDestroy(exe) == 0
