"""Scratch memory of device.cpp against a stand-in for the runtime, without a
GPU.

A failed device allocation that the library answers itself (a fallback without
scratch memory, a message to the caller) leaves no error behind: the HIP
runtime keeps a thread's last error until it is read, and the check after the
next kernel launch would report it as that launch's.

Scratch memory of a call that a graph records is that graph's until the graph
and its executables are gone: no other call gets it, and clearing the pool
does not free it."""
import os
import subprocess

import pytest

from tests.conftest import REPO

CSRC = os.path.join(REPO, "inference_c_amd", "csrc")
HIP_INCLUDE = "/opt/rocm/include"

RUNTIME = r"""
#include "kernels.hpp"
#include "pinned.hpp"
#include "sdk.hpp"
#include "tensor_device.h"
#include <cstdio>
#include <cstdlib>
#include <set>

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
static bool no_memory = false, capturing = false, no_retain = false;
static std::set<void *> memory;        // allocated and not freed
static void (*on_end)(void *) = nullptr;
static void *owned = nullptr;          // what the graph being captured retains
hipError_t hipMalloc(void **p, size_t n) {
    *p = no_memory ? nullptr : std::malloc(n);
    if (*p) memory.insert(*p);
    return *p ? hipSuccess : leave(hipErrorOutOfMemory);
}
hipError_t hipHostMalloc(void **p, size_t, unsigned) { *p = nullptr; return leave(hipErrorOutOfMemory); }
hipError_t hipFree(void *p) { memory.erase(p); std::free(p); return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
    *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamGetCaptureInfo_v2(hipStream_t, hipStreamCaptureStatus *s, unsigned long long *, hipGraph_t *g,
                                      const hipGraphNode_t **, size_t *) {
    *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    *g = reinterpret_cast<hipGraph_t>(&memory);
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) { return hipSuccess; }
hipError_t hipUserObjectCreate(hipUserObject_t *o, void *p, hipHostFn_t f, unsigned, unsigned) {
    on_end = f;
    *o = reinterpret_cast<hipUserObject_t>(p);
    return hipSuccess;
}
hipError_t hipUserObjectRelease(hipUserObject_t o, unsigned) { on_end(o); return hipSuccess; }
hipError_t hipGraphRetainUserObject(hipGraph_t, hipUserObject_t o, unsigned, unsigned) {
    if (no_retain) return leave(hipErrorInvalidValue);
    owned = o;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
}
namespace icsdk {
bool pinned_to_device(void *, const void *, size_t, hipStream_t, char *, size_t) { return true; }
bool pinned_to_host(void *, const void *, size_t, hipStream_t, char *, size_t) { return true; }
namespace k { size_t grid_reduce_scratch_bytes() { return 64; } }
}

"""

FAILURES = r"""
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
    no_memory = true;
    check("scratch", scratch_acquire(1 << 20) == nullptr);
    { ScratchBlock block(100); check("scratch block", block.get() == nullptr); }
    capturing = true;
    { ScratchBlock block(100); check("graph block", block.get() == nullptr); }
    no_memory = false;
    no_retain = true;
    { ScratchBlock block(100); check("graph that takes nothing", block.get() == nullptr); }
    no_memory = true;
    capturing = false;
    check("weight cache", weight_cache_get(text, sizeof text) == nullptr);
    check("host word", host_word_acquire() == nullptr);
    check("partials", grid_reduce_partials(text, sizeof text) == nullptr);
    TensorDeviceBuffer *buffer = nullptr;
    check("buffer", tensor_device_buffer_create(100, &buffer, text, sizeof text) == 0);
    return 0;
}
"""

GRAPH = r"""
#define CHECK(x) do { if (!(x)) { std::printf("%d: %s\n", __LINE__, #x); return 1; } } while (0)
int main() {
    using namespace icsdk;
    char text[128] = "";
    if (!sdk_ready(text, sizeof text)) return 2;
    void *first, *eager;
    { ScratchBlock block(5000); eager = block.get(); }
    capturing = true;
    { ScratchBlock block(5000); first = block.get(); }
    CHECK(first != nullptr && first != eager && owned != nullptr);
    void *const graph = owned;
    { ScratchBlock block(5000); CHECK(block.get() != first && block.get() != eager); }
    capturing = false;
    // calls between the replays, and a cleared pool
    { ScratchBlock a(5000), b(5000); CHECK(a.get() != first && b.get() != first); }
    scratch_clear();
    CHECK(memory.count(first) == 1 && memory.count(eager) == 0);
    // the graph is gone: the next capture takes the block, calls never do
    on_end(graph);
    { ScratchBlock a(5000); CHECK(a.get() != first); }
    capturing = true;
    { ScratchBlock block(5000); CHECK(block.get() == first); }
    capturing = false;
    on_end(owned);
    scratch_clear();
    CHECK(memory.count(first) == 0);
    return 0;
}
"""


@pytest.mark.parametrize("program", [FAILURES, GRAPH], ids=["failures", "graph"])
def test_scratch(tmp_path, program):
    if not os.path.isdir(os.path.join(HIP_INCLUDE, "hip")):
        pytest.skip("HIP headers absent")
    source, exe = tmp_path / "program.cpp", tmp_path / "program"
    source.write_text(RUNTIME + program)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-isystem", HIP_INCLUDE, "-I", CSRC,
                    "-I", os.path.join(REPO, "include"), "-o", str(exe), str(source),
                    os.path.join(CSRC, "device.cpp"), "-pthread"], check=True)
    result = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert result.returncode == 0, result.stdout
