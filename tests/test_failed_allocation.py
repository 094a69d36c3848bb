"""A failed device allocation that the library answers itself (a fallback
without scratch memory, a message to the caller) leaves no error behind: the
HIP runtime keeps a thread's last error until it is read, and the check after
the next kernel launch would report it as that launch's. device.cpp against a
stand-in for the runtime, without a GPU."""
import os
import subprocess

import pytest

from tests.conftest import REPO

CSRC = os.path.join(REPO, "inference_c_amd", "csrc")
HIP_INCLUDE = "/opt/rocm/include"

PROGRAM = r"""
#include "kernels.hpp"
#include "pinned.hpp"
#include "sdk.hpp"
#include "tensor_device.h"
#include <cstdio>
#include <cstdlib>

static hipError_t last = hipSuccess;   // as the runtime: kept until read
static hipError_t leave(hipError_t e) { if (e != hipSuccess) last = e; return e; }

extern "C" {
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return "out of memory"; }
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = nullptr; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t) { *p = nullptr; return leave(hipErrorOutOfMemory); }
hipError_t hipHostMalloc(void **p, size_t, unsigned) { *p = nullptr; return leave(hipErrorOutOfMemory); }
hipError_t hipFree(void *) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
}
namespace icsdk {
bool pinned_to_device(void *, const void *, size_t, hipStream_t, char *, size_t) { return true; }
bool pinned_to_host(void *, const void *, size_t, hipStream_t, char *, size_t) { return true; }
namespace k { size_t grid_reduce_scratch_bytes() { return 64; } }
}

static void check(const char *what, bool failed) {
    if (!failed || last != hipSuccess) {
        std::printf("%s: %s\n", what, failed ? "error left behind" : "did not fail");
        std::exit(1);
    }
}

int main() {
    using namespace icsdk;
    char text[128] = "";
    if (!sdk_ready(text, sizeof text)) return 2;
    check("scratch", scratch_acquire(1 << 20) == nullptr);
    { ScratchBlock block(100); check("scratch block", block.get() == nullptr); }
    check("weight cache", weight_cache_get(text, sizeof text) == nullptr);
    check("host word", host_word_acquire() == nullptr);
    check("partials", grid_reduce_partials(text, sizeof text) == nullptr);
    TensorDeviceBuffer *buffer = nullptr;
    check("buffer", tensor_device_buffer_create(100, &buffer, text, sizeof text) == 0);
    return 0;
}
"""


def test_answered_failures_leave_no_error(tmp_path):
    if not os.path.isdir(os.path.join(HIP_INCLUDE, "hip")):
        pytest.skip("HIP headers absent")
    source, exe = tmp_path / "program.cpp", tmp_path / "program"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-isystem", HIP_INCLUDE, "-I", CSRC,
                    "-I", os.path.join(REPO, "include"), "-o", str(exe), str(source),
                    os.path.join(CSRC, "device.cpp"), "-pthread"], check=True)
    result = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert result.returncode == 0, result.stdout
