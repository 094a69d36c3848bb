// Whole-tensor reductions for gfx950: sum+max of an f32 tensor and argmax.
//
// Two passes (one for a tensor that one block holds). Pass 1 (sum+max): block
// b streams the b-th contiguous chunk of 16-byte vectors, VPL vectors in
// flight per lane per step; the chunk grows with the tensor
// (sum_max_chunk_for). One-shot chunks measured ~15% faster on MI355X than a
// persistent grid-stride loop (88% vs 76% of HBM peak reading 4 GiB). For
// large tensors 32 vectors x 8 steps per lane (1 MiB chunks, 150 VGPRs, 3 waves per SIMD)
// ran 2^30 f32 in 606.2-606.8 us, 32 x 4 in 607.7-609.7 and 8 x 16 (8 waves
// per SIMD) in 612.1-613.5; 32 x 16 and 32 x 32 slower again. Past
// kMaxPartials chunks the grid strides over chunks. Each lane folds every
// 32 values (8 vectors) in f32 and adds that total to an f64 accumulator, so
// the rounding error stays near 32 f32 ulps of the group magnitude regardless
// of the tensor size. Lanes combine through shuffles, waves through LDS, and
// each block writes one partial. Pass 2: one 1024-lane block loads all
// partials at once, folds them in f64 and writes the result. No atomics and
// no counters, so the partial buffer needs no clearing between calls.
#include "kern_common.hpp"
#include "kernels.hpp"

#include <mutex>

namespace icsdk {
namespace {

constexpr int kPartials = 2048;     // argmax pass-1 grid
constexpr int kUnroll = 4;          // argmax vectors in flight per lane
// sum+max chunk of a pass-1 block, in vectors: VPL per lane in flight x steps
template <int VPL, int STEPS> constexpr size_t chunk_vectors() { return (size_t)kBlock * VPL * STEPS; }
constexpr size_t kChunkSmall = chunk_vectors<8, 1>();    // 32 KiB of f32
constexpr size_t kChunkMid = chunk_vectors<8, 4>();      // 128 KiB
constexpr size_t kChunkLarge = chunk_vectors<32, 8>();   // 1 MiB
constexpr int kMaxPartials = 4096;  // sum+max pass-1 grid cap (4 GiB per sweep: 2^30 f32 one-shot)
constexpr int kFoldBlock = 1024;    // pass-2 lanes
// sum+max of at most this many vectors: one block, one launch
constexpr size_t kOneBlockVectors = (size_t)kFoldBlock * 8;

struct Partial {
    double sum;
    float max;      // NaN when any element was NaN
    uint32_t index; // argmax: index of the block's best value (kNone if none)
};
constexpr uint32_t kNone = 0xffffffffu;

// ---- sum + max -------------------------------------------------------------

__device__ inline void fold(const f32x4 &v, float &group, float &m, bool &nan) {
    group += (v.x + v.y) + (v.z + v.w);
    m = fmaxf(fmaxf(m, fmaxf(v.x, v.y)), fmaxf(v.z, v.w));
    nan |= (v.x != v.x) | (v.y != v.y) | (v.z != v.z) | (v.w != v.w);
}

// One chunk: kSteps steps of kVpl coalesced vectors per lane of a block of
// kThreads. kGuard: the chunk runs past nvec (the last one), so vectors past
// the end are skipped.
template <bool kGuard, int kVpl, int kSteps, int kThreads = kBlock>
__device__ inline void sum_max_chunk(const f32x4 *__restrict__ xv, size_t first, size_t nvec,
                                     double &total, float &m, bool &nan) {
    static_assert(kVpl % 8 == 0, "whole f32 groups of 8 vectors");
#pragma unroll 1
    for (int step = 0; step < kSteps; ++step) {
        const size_t base = first + (size_t)step * kVpl * kThreads + threadIdx.x;
        f32x4 v[kVpl];
#pragma unroll
        for (int u = 0; u < kVpl; ++u) {
            const size_t i = base + (size_t)u * kThreads;
            if constexpr (kGuard) {
                v[u] = __builtin_nontemporal_load(xv + (i < nvec ? i : 0));
            } else {
                v[u] = __builtin_nontemporal_load(xv + i);
            }
        }
        // groups of 8 vectors (32 values) fold in f32, each into the f64 total
#pragma unroll
        for (int g = 0; g < kVpl / 8; ++g) {
            float group = 0.0f;
#pragma unroll
            for (int u = 8 * g; u < 8 * g + 8; ++u) {
                if constexpr (kGuard) {
                    if (base + (size_t)u * kThreads >= nvec) continue;
                }
                fold(v[u], group, m, nan);
            }
            total += (double)group;
        }
    }
}

// The block's totals: lanes by DPP, waves through LDS, then the first wave's
// lanes hold one wave each. Returns them in every lane of the first wave.
template <int kThreads>
__device__ inline Partial block_total(double total, float m, bool nan) {
    constexpr int W = kThreads / kWave;
    __shared__ double lds_sum[W];
    __shared__ float lds_max[W];
    total = wave_sum_f64(total);
    m = wave_max(m);
    if (wave_any(nan)) m = __builtin_nanf("");
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (lane == 0) {
        lds_sum[wave] = total;
        lds_max[wave] = m;
    }
    __syncthreads();
    if (wave != 0) return Partial{};
    const float wm = lane < W ? lds_max[lane < W ? lane : 0] : -__builtin_inff();
    total = wave_sum_f64(lane < W ? lds_sum[lane < W ? lane : 0] : 0.0);
    m = wave_max(wm);
    return Partial{total, wave_any(wm != wm) ? __builtin_nanf("") : m, 0};
}

// The elements after the last whole vector (fewer than 4).
__device__ inline void sum_max_tail(const float *x, size_t nvec, size_t n, double &total, float &m,
                                    bool &nan) {
    if (threadIdx.x < n - nvec * 4) {
        const float v = x[nvec * 4 + threadIdx.x];
        total += (double)v;
        m = fmaxf(m, v);
        nan |= v != v;
    }
}

template <int VPL, int STEPS>
__global__ __launch_bounds__(kBlock) void sum_max_pass1(const float *__restrict__ x,
                                                        size_t nvec, size_t n,
                                                        Partial *__restrict__ partials) {
    constexpr size_t kChunk = chunk_vectors<VPL, STEPS>();
    const f32x4 *xv = reinterpret_cast<const f32x4 *>(x);
    double total = 0.0;
    float m = -__builtin_inff();
    bool nan = false;
    for (size_t chunk = blockIdx.x; chunk * kChunk < nvec; chunk += gridDim.x) {
        const size_t first = chunk * kChunk;
        if (first + kChunk <= nvec) sum_max_chunk<false, VPL, STEPS>(xv, first, nvec, total, m, nan);
        else sum_max_chunk<true, VPL, STEPS>(xv, first, nvec, total, m, nan);
    }
    if (blockIdx.x == 0) sum_max_tail(x, nvec, n, total, m, nan);
    const Partial p = block_total<kBlock>(total, m, nan);
    if (threadIdx.x == 0) partials[blockIdx.x] = p;
}

// At most kOneBlockVectors vectors: the whole reduction in one block.
__global__ __launch_bounds__(kFoldBlock) void sum_max_one_block(const float *__restrict__ x,
                                                                size_t nvec, size_t n,
                                                                double *sum_out, float *max_out) {
    double total = 0.0;
    float m = -__builtin_inff();
    bool nan = false;
    if (nvec != 0)
        sum_max_chunk<true, 8, 1, kFoldBlock>(reinterpret_cast<const f32x4 *>(x), 0, nvec, total, m, nan);
    sum_max_tail(x, nvec, n, total, m, nan);
    const Partial p = block_total<kFoldBlock>(total, m, nan);
    if (threadIdx.x == 0) {
        if (sum_out) *sum_out = p.sum;
        if (max_out) *max_out = p.max;
    }
}

// count <= kPer * kFoldBlock: every lane's partials are requested before any
// is folded.
template <int kPer>
__global__ __launch_bounds__(kFoldBlock) void sum_max_pass2(const Partial *__restrict__ partials,
                                                            int count, double *sum_out,
                                                            float *max_out) {
    Partial p[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = (int)threadIdx.x + j * kFoldBlock;
        p[j] = partials[i < count ? i : 0];
    }
    double s = 0.0;
    float m = -__builtin_inff();
    bool nan = false;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        if ((int)threadIdx.x + j * kFoldBlock >= count) continue;
        s += p[j].sum;
        m = fmaxf(m, p[j].max);
        nan |= p[j].max != p[j].max;
    }
    const Partial t = block_total<kFoldBlock>(s, m, nan);
    if (threadIdx.x == 0) {
        if (sum_out) *sum_out = t.sum;
        if (max_out) *max_out = t.max;
    }
}

// ---- argmax ------------------------------------------------------------------

// (value, index) with "greater value wins, equal value -> lower index wins";
// NaN never compares greater, so it never wins. kNone marks "nothing yet".
__device__ inline void better(float &bv, uint32_t &bi, float v, uint32_t i) {
    if (v > bv || (v == bv && i < bi)) {
        bv = v;
        bi = i;
    }
}

__device__ inline void wave_argmax(float &bv, uint32_t &bi) {
    for (int offset = 32; offset > 0; offset >>= 1) {
        const float ov = __shfl_xor(bv, offset, kWave);
        const uint32_t oi = __shfl_xor(bi, offset, kWave);
        better(bv, bi, ov, oi);
    }
}

template <typename S>
__global__ __launch_bounds__(kBlock) void argmax_pass1(const S *__restrict__ x, size_t n,
                                                       Partial *__restrict__ partials) {
    __shared__ float lds_v[kBlock / kWave];
    __shared__ uint32_t lds_i[kBlock / kWave];
    constexpr int E = Vec16<S>::N;
    const size_t nvec = n / E;
    const size_t stride = (size_t)gridDim.x * kBlock;
    float bv = -__builtin_inff();
    uint32_t bi = kNone;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < nvec; i += stride) {
        const Vec16<S> v = load16_stream(x + i * E);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const float f = Elem<S>::load(v.v[e]);
            if (f > bv) {  // strict: within one lane indices ascend
                bv = f;
                bi = (uint32_t)(i * E + e);
            }
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < n - nvec * E) {
        const uint32_t t = (uint32_t)(nvec * E + threadIdx.x);
        better(bv, bi, Elem<S>::load(x[t]), t);
    }
    wave_argmax(bv, bi);
    const int wave = threadIdx.x / kWave;
    if ((threadIdx.x & (kWave - 1)) == 0) {
        lds_v[wave] = bv;
        lds_i[wave] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / kWave; ++w) better(bv, bi, lds_v[w], lds_i[w]);
        partials[blockIdx.x] = Partial{0.0, bv, bi};
    }
}

template <typename S>
__global__ __launch_bounds__(kBlock) void argmax_pass2(const S *__restrict__ x,
                                                       const Partial *__restrict__ partials,
                                                       int count, uint32_t *index_out) {
    __shared__ float lds_v[kBlock / kWave];
    __shared__ uint32_t lds_i[kBlock / kWave];
    float bv = -__builtin_inff();
    uint32_t bi = kNone;
    constexpr int kPer = kPartials / kBlock;   // requested before any is compared
    float pv[kPer];
    uint32_t pi[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = (int)threadIdx.x + j * kBlock;
        pv[j] = partials[i < count ? i : 0].max;
        pi[j] = partials[i < count ? i : 0].index;
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) better(bv, bi, pv[j], pi[j]);
    wave_argmax(bv, bi);
    const int wave = threadIdx.x / kWave;
    if ((threadIdx.x & (kWave - 1)) == 0) {
        lds_v[wave] = bv;
        lds_i[wave] = bi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / kWave; ++w) better(bv, bi, lds_v[w], lds_i[w]);
        const float first = Elem<S>::load(x[0]);
        // The reference scans from element 0 with a strict '>': a NaN first
        // element is never replaced, and when the largest non-NaN value is
        // -inf (or there is none) element 0 is never beaten either.
        *index_out = (first != first || bi == kNone || bv == -__builtin_inff()) ? 0u : bi;
    }
}

// At most kArgOneBlock vectors: one block, one launch (1000 f16: 6.2 -> 3.8 us
// per call, 65536 f16 6.4 -> 4.8).
constexpr size_t kArgOneBlock = (size_t)kFoldBlock * 8;
template <typename S>
__global__ __launch_bounds__(kFoldBlock) void argmax_one_block(const S *__restrict__ x, size_t n,
                                                               uint32_t *index_out) {
    constexpr int W = kFoldBlock / kWave, E = Vec16<S>::N;
    __shared__ float lds_v[W];
    __shared__ uint32_t lds_i[W];
    const uint32_t nvec = (uint32_t)(n / E);
    float bv = -__builtin_inff();
    uint32_t bi = kNone;
    if (nvec != 0) {
        Vec16<S> v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const uint32_t i = threadIdx.x + u * kFoldBlock;
            v[u] = load16_stream(x + (size_t)(i < nvec ? i : 0) * E);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const uint32_t i = threadIdx.x + u * kFoldBlock;
            if (i >= nvec) continue;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const float f = Elem<S>::load(v[u].v[e]);
                if (f > bv) {  // strict: within one lane indices ascend
                    bv = f;
                    bi = i * E + e;
                }
            }
        }
    }
    if (threadIdx.x < n - (size_t)nvec * E) {
        const uint32_t t = nvec * E + threadIdx.x;
        better(bv, bi, Elem<S>::load(x[t]), t);
    }
    wave_argmax(bv, bi);
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (lane == 0) {
        lds_v[wave] = bv;
        lds_i[wave] = bi;
    }
    __syncthreads();
    if (wave != 0) return;
    bv = lane < W ? lds_v[lane < W ? lane : 0] : -__builtin_inff();
    bi = lane < W ? lds_i[lane < W ? lane : 0] : kNone;
    wave_argmax(bv, bi);
    if (lane == 0) {
        const float first = Elem<S>::load(x[0]);   // (the rule of argmax_pass2)
        *index_out = (first != first || bi == kNone || bv == -__builtin_inff()) ? 0u : bi;
    }
}

inline int pass1_grid(size_t work) {
    const size_t blocks = (work + (size_t)kBlock * kUnroll - 1) / ((size_t)kBlock * kUnroll);
    return blocks < 1 ? 1 : (blocks > (size_t)kPartials ? kPartials : (int)blocks);
}

}  // namespace
}  // namespace icsdk

// Partials of the allocation-free sum+max (tensor_sum_max_f32_no_alloc): one
// Partial per pass-1 block, and the pass-1 grid never exceeds kMaxPartials
// blocks (past that the blocks stride over chunks), so 64 KiB covers every
// input size. Each device the library runs on holds its own copy until the
// process ends. Host code never passes this name to a kernel: its device
// address comes from hipGetSymbolAddress, once per device.
static __device__ __align__(256) unsigned char
    scratch[sizeof(icsdk::Partial) * icsdk::kMaxPartials];

namespace icsdk {
namespace k {

size_t no_alloc_scratch_bytes() { return sizeof(scratch); }

hipError_t no_alloc_scratch(void **ptr) {
    constexpr int kMaxDevices = 64;
    static std::mutex lookup;
    static void *address[kMaxDevices] = {};
    *ptr = nullptr;
    int device = -1;
    hipError_t status = hipGetDevice(&device);
    if (status != hipSuccess) return status;
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(lookup);
    if (address[device] == nullptr) {
        void *found = nullptr;
        status = hipGetSymbolAddress(&found, HIP_SYMBOL(scratch));
        if (status != hipSuccess) return status;
        address[device] = found;
    }
    *ptr = address[device];
    return hipSuccess;
}

// Pass-1 chunk for nvec vectors: 32 KiB up to 1024 blocks (32 MiB), 128 KiB until
// 1 MiB chunks give every CU a block (256 MiB). Small tensors need many short
// blocks to fill the chip, large ones few long ones (us per call in a row on
// one tensor, 1 MiB chunks everywhere -> here: 1000 f32 12.5 -> 3.8 (one block),
// 2^20 20.5 -> 7.2, 2^22 25.4 -> 7.2 (another tensor each time 8.0), 2^24 28.4 ->
// 13.8, 2^25 + 4 29.0 -> 22.5, 2^26 - 4 44.0 -> 42.1; 3 x 2^24 the same; at 2^26
// 128 KiB chunks 42.0, 1 MiB 41.6).
static size_t sum_max_chunk_for(size_t nvec) {
    if (nvec <= kChunkSmall * 1024) return kChunkSmall;
    if (nvec < kChunkLarge * 256) return kChunkMid;
    return kChunkLarge;
}

size_t sum_max_partials_bytes(size_t n) {
    const size_t chunk = sum_max_chunk_for(n / 4);
    const size_t chunks = (n / 4 + chunk - 1) / chunk;
    const size_t grid = chunks < 1 ? 1 : (chunks > (size_t)kMaxPartials ? kMaxPartials : chunks);
    return grid * sizeof(Partial);
}

hipError_t sum_max_f32_no_alloc(const float *x, size_t n, double *sum_out, float *max_out,
                                void *scratch_ptr, size_t scratch_bytes, hipStream_t s) {
    if (n == 0 || ((uintptr_t)x & 15u) != 0 || scratch_ptr == nullptr ||
        sum_max_partials_bytes(n) > scratch_bytes)
        return hipErrorInvalidValue;
    return sum_max_f32(x, n, sum_out, max_out, scratch_ptr, s);
}


size_t grid_reduce_scratch_bytes() {
    return sizeof(Partial) * (kMaxPartials > kPartials ? kMaxPartials : kPartials);
}

hipError_t sum_max_f32(const float *x, size_t n, double *sum_out, float *max_out,
                       void *partials, hipStream_t s) {
    if (n == 0) return hipErrorInvalidValue;
    if (((uintptr_t)x & 15u) != 0) return hipErrorInvalidValue;
    const size_t nvec = n / 4;
    const int grid = (int)(sum_max_partials_bytes(n) / sizeof(Partial));
    auto *p = static_cast<Partial *>(partials);
    if (nvec <= kOneBlockVectors) {
        hipLaunchKernelGGL(sum_max_one_block, dim3(1), dim3(kFoldBlock), 0, s, x, nvec, n, sum_out,
                           max_out);
        return hipGetLastError();
    }
    const size_t chunk = sum_max_chunk_for(nvec);
    if (chunk == kChunkSmall)
        hipLaunchKernelGGL((sum_max_pass1<8, 1>), dim3(grid), dim3(kBlock), 0, s, x, nvec, n, p);
    else if (chunk == kChunkMid)
        hipLaunchKernelGGL((sum_max_pass1<8, 4>), dim3(grid), dim3(kBlock), 0, s, x, nvec, n, p);
    else
        hipLaunchKernelGGL((sum_max_pass1<32, 8>), dim3(grid), dim3(kBlock), 0, s, x, nvec, n, p);
    if (grid <= kFoldBlock)
        hipLaunchKernelGGL((sum_max_pass2<1>), dim3(1), dim3(kFoldBlock), 0, s, p, grid, sum_out,
                           max_out);
    else
        hipLaunchKernelGGL((sum_max_pass2<kMaxPartials / kFoldBlock>), dim3(1), dim3(kFoldBlock), 0,
                           s, p, grid, sum_out, max_out);
    return hipGetLastError();
}

template <typename S>
hipError_t argmax_launch(const S *x, size_t n, uint32_t *index_out, void *partials,
                         hipStream_t s) {
    if (n == 0 || n > 0xffffffffu || ((uintptr_t)x & 15u) != 0) return hipErrorInvalidValue;
    if (n / Vec16<S>::N <= kArgOneBlock) {
        hipLaunchKernelGGL((argmax_one_block<S>), dim3(1), dim3(kFoldBlock), 0, s, x, n, index_out);
        return hipGetLastError();
    }
    const int grid = pass1_grid(n / Vec16<S>::N);
    auto *p = static_cast<Partial *>(partials);
    hipLaunchKernelGGL((argmax_pass1<S>), dim3(grid), dim3(kBlock), 0, s, x, n, p);
    hipLaunchKernelGGL((argmax_pass2<S>), dim3(1), dim3(kBlock), 0, s, x, p, grid, index_out);
    return hipGetLastError();
}

hipError_t argmax_f32(const float *x, size_t n, uint32_t *index_out, void *partials,
                      hipStream_t s) {
    return argmax_launch<float>(x, n, index_out, partials, s);
}

hipError_t argmax_f16(const uint16_t *x, size_t n, uint32_t *index_out, void *partials,
                      hipStream_t s) {
    return argmax_launch<_Float16>(reinterpret_cast<const _Float16 *>(x), n, index_out,
                                   partials, s);
}

}  // namespace k
}  // namespace icsdk
