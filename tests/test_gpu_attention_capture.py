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
