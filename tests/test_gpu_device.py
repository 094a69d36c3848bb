"""Device buffers and the asynchronous contract, following the reference's
tests/test_tensor_device.c: storage contract, 16 MiB upload/copy/download
round trip in a 64 MiB working set, asynchronous F16 residual add checked
bit-exact, and backend selection through TENSOR_BACKEND."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TEST_BYTES = 16 * 1024 * 1024
WORKING_SET = TEST_BYTES * 4


def test_storage_contract(sdk):
    t = sdk.tensor("u8", (WORKING_SET,))
    assert sdk.lib.tensor_buffer_storage(t.handle) == 1
    assert sdk.lib.tensor_buffer_data(t.handle) is None
    assert sdk.lib.tensor_buffer_byte_length(t.handle) == WORKING_SET
    assert t.device_ptr() % 256 == 0
    empty = sdk.tensor("f16", (0,))
    assert empty.device_ptr() == 0  # zero-byte device tensors allocate nothing


def test_round_trip_through_device_copy(sdk):
    # test_tensor_device.c:82-113
    i = np.arange(WORKING_SET, dtype=np.uint64)
    pattern = ((i * 131 + (i >> 8) + 17) & 0xFF).astype(np.uint8)
    src = sdk.tensor("u8", (WORKING_SET,))
    dst = sdk.tensor("u8", (WORKING_SET,))
    err = ctypes.create_string_buffer(256)
    assert sdk.lib.tensor_buffer_upload(src.handle, 0, pattern.ctypes.data, TEST_BYTES, err, 256), err.value
    assert sdk.lib.tensor_buffer_copy_device(dst.handle, 0, src.handle, 0, TEST_BYTES, err, 256), err.value
    sdk.synchronize()
    back = np.empty(TEST_BYTES, np.uint8)
    assert sdk.lib.tensor_buffer_download(dst.handle, 0, back.ctypes.data, TEST_BYTES, err, 256), err.value
    assert np.array_equal(back, pattern[:TEST_BYTES])
    # offset copy inside the working set, and range checks
    assert sdk.lib.tensor_buffer_copy_device(dst.handle, 3 * TEST_BYTES + 5, src.handle, 7, 1000, err, 256)
    part = np.empty(1000, np.uint8)
    assert sdk.lib.tensor_buffer_download(dst.handle, 3 * TEST_BYTES + 5, part.ctypes.data, 1000, err, 256)
    assert np.array_equal(part, pattern[7:1007])
    assert not sdk.lib.tensor_buffer_copy_device(dst.handle, WORKING_SET - 4, src.handle, 0, 8, err, 256)
    assert err.value == b"tensor device copy requires valid device-resident ranges"


def test_async_residual_add_exact(sdk):
    # test_tensor_device.c:144-176
    left = np.array([0x3c00, 0xc000, 0x4200, 0xc400], np.uint16).view(np.float16)
    right = np.array([0x4000, 0x3800, 0xbc00, 0x4400], np.uint16).view(np.float16)
    tl, tr, to = sdk.from_numpy(left), sdk.from_numpy(right), sdk.tensor("f16", (4,))
    sdk.call("tensor_residual_add_f16", tl, tr, to)
    sdk.synchronize()
    assert to.download().view(np.uint16).tolist() == [0x4200, 0xbe00, 0x4000, 0x0000]


def test_mixed_storage_rejected(sdk):
    h = sdk.tensor("f16", (4,), device=False)
    d = sdk.tensor("f16", (4,))
    ok, msg = sdk.try_call("tensor_residual_add_f16", h, d, d)
    assert not ok and msg == "F16 residual add operands must use the same storage type"
    ok, msg = sdk.try_call("tensor_silu_f16", h, d)
    assert not ok and msg == "SiLU operands must use the same storage type"


def test_backend_selection(sdk, monkeypatch):
    lib = sdk.lib
    for value in (None, "", "auto", "hip"):
        if value is None:
            monkeypatch.delenv("TENSOR_BACKEND", raising=False)
        else:
            monkeypatch.setenv("TENSOR_BACKEND", value)
        p = lib.tensor_compute_preferred_backend()
        assert p and ctypes.cast(p, ctypes.POINTER(ctypes.c_char_p))[0] == b"hip"
    a = sdk.from_numpy(np.ones(8, np.float16))
    for value in ("cuda", "metal", "qnn", "bogus"):
        monkeypatch.setenv("TENSOR_BACKEND", value)
        assert lib.tensor_compute_preferred_backend() is None
        # the reference routes the device residual add through the preferred
        # backend (tensor_ops.c:596-605): with none selected it fails
        ok, msg = sdk.try_call("tensor_residual_add_f16", a, a, a)
        assert not ok and msg == "device F16 residual add backend operation failed"
    monkeypatch.delenv("TENSOR_BACKEND")
    sdk.call("tensor_residual_add_f16", a, a, a)
    assert np.all(a.download() == 2)


def test_stream_is_exposed(sdk):
    assert sdk.stream() != 0


# ---- pinned staging ----------------------------------------------------------
# Host memory crosses PCIe through 4 MiB page-locked chunks (at most three per
# transfer, reused in rotation). Sizes below straddle every chunk boundary
# case: sub-chunk, exactly one chunk, one chunk plus a tail, several chunks
# reusing the same three.

STAGING_SIZES = [1, 4095, (1 << 20) + 1, 4 << 20, (4 << 20) + 3, (13 << 20) + 7, (9 << 20) + 1, 40 << 20]


@pytest.mark.parametrize("nbytes", STAGING_SIZES)
def test_pinned_round_trip(sdk, nbytes):
    rng = np.random.default_rng(nbytes)
    data = rng.integers(0, 256, nbytes, dtype=np.uint8)
    t = sdk.tensor("u8", (nbytes,)).upload(data)
    data_copy = data.copy()
    data[:] = 0  # the upload has consumed the source when it returns
    assert np.array_equal(t.download(), data_copy)


def test_pinned_upload_at_offsets(sdk):
    """Uploads and downloads of sub-ranges at odd offsets."""
    rng = np.random.default_rng(7)
    total = (9 << 20) + 5
    t = sdk.tensor("u8", (total,))
    want = np.zeros(total, np.uint8)
    t.upload(want)
    err = ctypes.create_string_buffer(256)
    for offset, length in ((3, 17), (1 << 20, (5 << 20) + 1), (total - 9, 9), (0, total)):
        part = rng.integers(0, 256, length, dtype=np.uint8)
        assert sdk.lib.tensor_buffer_upload(t.handle, offset, part.ctypes.data, length, err, 256)
        want[offset:offset + length] = part
        got = np.empty(length, np.uint8)
        assert sdk.lib.tensor_buffer_download(t.handle, offset, got.ctypes.data, length, err, 256)
        assert np.array_equal(got, part)
    assert np.array_equal(t.download(), want)


def test_host_slots_from_several_threads(sdk, orc):
    """Host-pointer slots called concurrently from 4 threads, each moving
    several chunks per call: every result matches the oracle bit for bit."""
    import threading
    from tests.test_gpu_vtable import Table
    table = ctypes.cast(sdk.lib.tensor_compute_hip_backend(), ctypes.POINTER(Table)).contents
    fn = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_void_p,
                          ctypes.c_size_t)(table.residual_add_f16)
    sizes = [(3 << 20) + 1, (6 << 20) + 11, 777, (9 << 20) + 3]
    inputs = [(orc.normal((n,), 80 + i, 0, 0.0, 1.0, "f16"), orc.normal((n,), 80 + i, 1, 0.0, 1.0, "f16"))
              for i, n in enumerate(sizes)]
    wants = [orc.add(a, b) for a, b in inputs]
    failures = []

    def work(i):
        a, b = inputs[i]
        for _ in range(3):
            y = np.empty_like(a)
            if not fn(a.ctypes.data, b.ctypes.data, y.ctypes.data, a.size):
                failures.append((i, "call failed"))
            elif not np.array_equal(y.view(np.uint16), wants[i].view(np.uint16)):
                failures.append((i, "wrong result"))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not failures, failures
    ctypes.CFUNCTYPE(None)(table.release_cache)()
    # the pool is rebuilt on the next call
    y = np.empty_like(inputs[0][0])
    assert fn(inputs[0][0].ctypes.data, inputs[0][1].ctypes.data, y.ctypes.data, sizes[0])
    assert np.array_equal(y.view(np.uint16), wants[0].view(np.uint16))


def test_calls_after_a_failed_creation(sdk, orc):
    """A tensor that device memory does not hold is refused with a message, and
    the next call is not refused for it."""
    from inference_c_amd.sdk import SdkError
    x = orc.normal((3, 70001), 84, 0, 0.0, 1.0, "f32")
    tx, ty = sdk.from_numpy(x), sdk.tensor("f32", x.shape)
    for _ in range(2):
        with pytest.raises(SdkError, match="out of memory"):
            sdk.tensor("f32", (1 << 48,))
        sdk.call("tensor_softmax_f32", tx, 0, ty)
        assert np.allclose(ty.download().sum(-1), 1.0, atol=1e-4)
