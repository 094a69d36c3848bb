// Linear layers of few input rows, and small ones: y[r][o] = sum_i x[r][i] w[o][i]
// (+ bias[o]) for f16 or f32 weights stored [out, in] row-major, the layout
// of the reference's tensor_linear_* (src/common/tensor_ops.c:318-398;
// the CUDA backend's cuBLAS call, tensor_compute_cuda.cu:174-265).
//
// At one to four input rows the product is a stream over the weights
// (2 or 4 bytes each, read once) with a few flops per byte, so it is written
// as a GEMV rather than handed to a GEMM library: a wave owns O output rows
// (O = 1 measured fastest) and walks them, each lane reading 16-byte vectors
// at a 64-vector (1 KiB) stride, so every load instruction reads 1 KiB of
// one weight row contiguously, kUnroll of them in flight. Lane l's slice of
// x (R rows) is loaded once per vector position and reused for the O rows.
// f16: v_dot2_f32_f16 (exact products, f32 sums); f32: fma. The lanes'
// partial sums are folded with DPP; the bias is added in f32 before the
// result is rounded to the output type. Bound: HBM bytes of the weights.
#include "kern_common.hpp"
#include "kernels.hpp"

namespace icsdk {
namespace k {
namespace {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
// 16 bytes at an element's alignment
template <typename T> using u32x4_any = uint32_t __attribute__((ext_vector_type(4), aligned(sizeof(T))));

constexpr int kUnroll = 4;   // vector positions in flight per lane

// sum of the products of one 16-byte vector of weights and of x
template <typename T>
__device__ inline float vec_dot(const u32x4 &w, const u32x4 &x, float acc) {
    if constexpr (sizeof(T) == 2) {
        // elements copied into scalars before the bit casts (a bit cast of a
        // vector element compiles to one of element 0)
        const uint32_t wa[4] = {w.x, w.y, w.z, w.w}, xa[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, wa[i]), __builtin_bit_cast(half2_t, xa[i]),
                                         acc, false);
    } else {
        const f32x4 wf = __builtin_bit_cast(f32x4, w), xf = __builtin_bit_cast(f32x4, x);
        acc = __builtin_fmaf(wf.x, xf.x, acc);
        acc = __builtin_fmaf(wf.y, xf.y, acc);
        acc = __builtin_fmaf(wf.z, xf.z, acc);
        acc = __builtin_fmaf(wf.w, xf.w, acc);
    }
    return acc;
}

// Grid: x = waves of O output rows (4 waves per block), y = groups of R
// input rows. Requires x, w 16-byte aligned and in a multiple of the
// elements per 16 bytes (every row then starts 16-byte aligned).
template <typename T, int R, int O>
__global__ __launch_bounds__(kBlock) void gemv_kernel(const T *__restrict__ x, const T *__restrict__ w,
                                                      const T *__restrict__ bias, T *__restrict__ y,
                                                      uint32_t rows, uint32_t in, uint32_t out) {
    constexpr uint32_t E = 16 / sizeof(T);
    const uint32_t lane = threadIdx.x & (kWave - 1);
    // the wave's index in the grid, formed without the work-item number
    // (blockIdx.x * kBlock), which would wrap in 32 bits for a large grid
    const uint32_t wave =
        __builtin_amdgcn_readfirstlane(blockIdx.x * (kBlock / kWave) + threadIdx.x / kWave);
    const uint32_t o0 = wave * O;
    if (o0 >= out) return;
    const uint32_t r0 = blockIdx.y * R;
    const uint32_t nvec = in / E;
    // rows past the end are clamped onto the last one (computed, not stored)
    const u32x4 *wrow[O];
    const u32x4 *xrow[R];
#pragma unroll
    for (int o = 0; o < O; ++o)
        wrow[o] = reinterpret_cast<const u32x4 *>(w + (size_t)min(o0 + o, out - 1) * in);
#pragma unroll
    for (int r = 0; r < R; ++r)
        xrow[r] = reinterpret_cast<const u32x4 *>(x + (size_t)min(r0 + r, rows - 1) * in);
    float acc[O][R];
#pragma unroll
    for (int o = 0; o < O; ++o)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[o][r] = 0.0f;

    constexpr uint32_t kStep = kWave * kUnroll;
    uint32_t v0 = 0;
    // whole steps: every lane's kUnroll vectors exist
    for (; v0 + kStep <= nvec; v0 += kStep) {
        u32x4 wv[kUnroll][O], xv[kUnroll][R];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const uint32_t v = v0 + kWave * u + lane;
#pragma unroll
            for (int o = 0; o < O; ++o) wv[u][o] = __builtin_nontemporal_load(wrow[o] + v);
#pragma unroll
            for (int r = 0; r < R; ++r) xv[u][r] = xrow[r][v];
        }
#pragma unroll
        for (int u = 0; u < kUnroll; ++u)
#pragma unroll
            for (int o = 0; o < O; ++o)
#pragma unroll
                for (int r = 0; r < R; ++r) acc[o][r] = vec_dot<T>(wv[u][o], xv[u][r], acc[o][r]);
    }
    // the rest, one vector position at a time
    for (uint32_t v = v0 + lane; v < nvec; v += kWave) {
#pragma unroll
        for (int o = 0; o < O; ++o) {
            const u32x4 wv = __builtin_nontemporal_load(wrow[o] + v);
#pragma unroll
            for (int r = 0; r < R; ++r) acc[o][r] = vec_dot<T>(wv, xrow[r][v], acc[o][r]);
        }
    }
#pragma unroll
    for (int o = 0; o < O; ++o) {
        const float b = bias != nullptr ? (float)bias[min(o0 + o, out - 1)] : 0.0f;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float total = wave_sum(acc[o][r]) + b;
            if (lane == 0 && o0 + o < out && r0 + r < rows) y[(size_t)(r0 + r) * out + o0 + o] = (T)total;
        }
    }
}

// Small products of more input rows (and rows no GEMV can read in whole
// vectors): each weight is used by more rows than v_dot2 carries for free, so
// the products go to MFMA. A block takes 16 OT output columns of 16 RG input
// rows; its NW waves share the k range, in interleaved runs of UN 128-byte lines
// per row, and their partial sums meet in LDS. The register layout of an MFMA
// operand has 16 rows in 16 neighbouring lanes: loaded so from memory, every
// quarter of a load instruction touches 16 lines (16 x 8192 -> 8192 f16 42 us).
// So 8 lanes read a row's line, the wave passes it through its own piece of LDS
// (16-byte vectors, the vector number xor-ed with the row: conflict-free both
// ways), and the next run's loads are in flight meanwhile. Lane (i, g) of the
// MFMA takes vector 4 c + g of row i as chunk c: the k order inside a chunk is
// the memory's, the same for both.
// Bound: a block's operands through its CU (x again for every 16 columns),
// a few memory latencies in a row, and the launch.
template <typename T, int RG, int OT, int NW, int UN>
__global__ __launch_bounds__(NW * kWave) void skinny_kernel(const T *__restrict__ x, const T *__restrict__ w,
                                                            const T *__restrict__ bias, T *__restrict__ y,
                                                            uint32_t rows, uint32_t in, uint32_t out) {
    constexpr uint32_t E = 16 / sizeof(T);
    constexpr uint32_t kLine = 8 * E;       // elements of a 128-byte line
    constexpr uint32_t kTiles = OT + RG;    // 16-row tiles of a run: weights, then x
    constexpr uint32_t kTileVecs = 16 * 8;  // 16-byte vectors of a tile's line
    __shared__ u32x4 stage[NW][UN * kTiles * kTileVecs];
    static_assert(UN * kTiles * kTileVecs >= OT * RG * kWave, "the partial sums fit the stages");
    const uint32_t lane = threadIdx.x & (kWave - 1), i = lane & 15, g = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t o0 = blockIdx.x * (16 * OT), r0 = blockIdx.y * (16 * RG);
    const uint32_t lr = lane / 8, lv = lane % 8;   // the row (and + 8) and the vector this lane loads
    // columns and rows past the end read the last one (computed, not stored)
    const T *row[kTiles][2];
#pragma unroll
    for (uint32_t t = 0; t < kTiles; ++t)
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h)
            row[t][h] = t < OT ? w + (size_t)min(o0 + 16 * t + 8 * h + lr, out - 1) * in
                               : x + (size_t)min(r0 + 16 * (t - OT) + 8 * h + lr, rows - 1) * in;
    f32x4 acc[OT][RG];
#pragma unroll
    for (int o = 0; o < OT; ++o)
#pragma unroll
        for (int r = 0; r < RG; ++r) acc[o][r] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    u32x4 reg[UN][kTiles][2];
    // Rows start at any element. A vector that the row's end cuts is read so
    // that it ends there, and the elements of the vector before it are zeroed
    // when staged (in x and w alike, so the k of both still agree); vectors
    // past the end likewise, as a whole.
    auto fetch = [&](uint32_t k) {
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const uint32_t at = min(k + u * kLine + lv * E, in - E);
#pragma unroll
            for (uint32_t t = 0; t < kTiles; ++t)
#pragma unroll
                for (uint32_t h = 0; h < 2; ++h) {
                    const u32x4_any<T> *p = reinterpret_cast<const u32x4_any<T> *>(row[t][h] + at);
                    reg[u][t][h] = t < OT ? __builtin_nontemporal_load(p) : *p;
                }
        }
    };
    auto put = [&](uint32_t k) {
        if (k + UN * kLine > in) {
#pragma unroll
            for (int u = 0; u < UN; ++u) {
                const uint32_t at = k + u * kLine + lv * E;
                const uint32_t drop = at + E <= in ? 0 : min(at + E - in, E) * sizeof(T);   // bytes from its start
                u32x4 keep;
#pragma unroll
                for (uint32_t d = 0; d < 4; ++d)
                    keep[d] = 4 * d >= drop ? 0xffffffffu : 4 * d + 2 >= drop ? 0xffff0000u : 0u;
#pragma unroll
                for (uint32_t t = 0; t < kTiles; ++t) {
                    reg[u][t][0] &= keep;
                    reg[u][t][1] &= keep;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < UN; ++u)
#pragma unroll
            for (uint32_t t = 0; t < kTiles; ++t)
#pragma unroll
                for (uint32_t h = 0; h < 2; ++h)
                    stage[wave][(u * kTiles + t) * kTileVecs + (8 * h + lr) * 8 + (lv ^ lr)] = reg[u][t][h];
    };
    constexpr uint32_t kRun = UN * kLine;
    uint32_t k = wave * kRun;
    if (k < in) fetch(k);
    while (k < in) {
        put(k);
        const uint32_t next = in - k > NW * kRun ? k + NW * kRun : in;
        if (next < in) fetch(next);
        // the stage is this wave's alone: only its own order matters
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
        for (int u = 0; u < UN; ++u)
#pragma unroll
            for (uint32_t c = 0; c < 2; ++c) {
                u32x4 f[kTiles];
#pragma unroll
                for (uint32_t t = 0; t < kTiles; ++t)
                    f[t] = stage[wave][(u * kTiles + t) * kTileVecs + i * 8 + ((4 * c + g) ^ (i & 7))];
#pragma unroll
                for (int o = 0; o < OT; ++o)
#pragma unroll
                    for (int r = 0; r < RG; ++r) {
                        if constexpr (sizeof(T) == 2) {
                            acc[o][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                                __builtin_bit_cast(half8, f[o]), __builtin_bit_cast(half8, f[OT + r]), acc[o][r], 0, 0, 0);
                        } else {
                            const f32x4 wf = __builtin_bit_cast(f32x4, f[o]), xf = __builtin_bit_cast(f32x4, f[OT + r]);
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                acc[o][r] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[e], xf[e], acc[o][r], 0, 0, 0);
                        }
                    }
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        k = next;
    }
#pragma unroll
    for (int o = 0; o < OT; ++o)
#pragma unroll
        for (int r = 0; r < RG; ++r) stage[wave][(o * RG + r) * kWave + lane] = __builtin_bit_cast(u32x4, acc[o][r]);
    __syncthreads();
    // tile t's element (lane, j): column o0 + 16 (t / RG) + 4 g + j, row r0 + 16 (t % RG) + i
    for (uint32_t t = wave; t < OT * RG; t += NW) {
        f32x4 sum = __builtin_bit_cast(f32x4, stage[0][t * kWave + lane]);
#pragma unroll
        for (int p = 1; p < NW; ++p) sum += __builtin_bit_cast(f32x4, stage[p][t * kWave + lane]);
        const uint32_t col = o0 + 16 * (t / RG) + 4 * g, r = r0 + 16 * (t % RG) + i;
        if (r >= rows) continue;
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j)
            if (col + j < out) y[(size_t)r * out + col + j] = (T)(sum[j] + (bias != nullptr ? (float)bias[col + j] : 0.0f));
    }
}

template <typename T, int R, int O>
hipError_t launch(const T *x, const T *w, const T *bias, T *y, size_t rows, size_t in, size_t out,
                  hipStream_t s) {
    constexpr size_t kWavesPerBlock = kBlock / kWave;
    const size_t waves = (out + O - 1) / O;
    const dim3 grid((unsigned)((waves + kWavesPerBlock - 1) / kWavesPerBlock), (unsigned)((rows + R - 1) / R));
    gemv_kernel<T, R, O><<<grid, kBlock, 0, s>>>(x, w, bias, y, (uint32_t)rows, (uint32_t)in, (uint32_t)out);
    return hipGetLastError();
}

template <typename T>
hipError_t gemv(const T *x, const T *w, const T *bias, T *y, size_t rows, size_t in, size_t out,
                hipStream_t s) {
    // one output row per wave (1 x 8192 -> 8192 f16: 21.9 us; 2 rows 22.5,
    // 4 rows 30.6; hipBLASLt 26.0)
    constexpr int O = 1;
    switch (rows) {
    case 1: return launch<T, 1, O>(x, w, bias, y, rows, in, out, s);
    case 2: return launch<T, 2, O>(x, w, bias, y, rows, in, out, s);
    case 3: return launch<T, 3, O>(x, w, bias, y, rows, in, out, s);
    default: return launch<T, 4, O>(x, w, bias, y, rows, in, out, s);
    }
}

template <typename T, int RG, int OT, int NW, int UN>
hipError_t launch_skinny(const T *x, const T *w, const T *bias, T *y, size_t rows, size_t in, size_t out,
                         hipStream_t s) {
    const dim3 grid((unsigned)((out + 16 * OT - 1) / (16 * OT)), (unsigned)((rows + 16 * RG - 1) / (16 * RG)));
    skinny_kernel<T, RG, OT, NW, UN>
        <<<grid, NW * kWave, 0, s>>>(x, w, bias, y, (uint32_t)rows, (uint32_t)in, (uint32_t)out);
    return hipGetLastError();
}

// Small products on skinny_kernel, or hipErrorNotSupported. The library's call
// is bound by its host part, 7.1 us one after another on one host and 8.4 on
// another, and streams large weights better. us per call here, the library's
// in brackets, calls in a row with other buffers each time on the faster host
// (a call that is waited for gains more: 16 x 4096 -> 4096 21.0 [24.5], 128 x
// 2048 -> 1000 17.8 [21.6], 100 x 3072 -> 200 19.0 [20.8]):
//   up to 32 input rows: f16 weights of rows of up to 8 KB, 34 MB in all (16 x
//   4096 -> 4096 8.7 [10.2], 32 x 4096 -> 4096 9.9 [12.7], 16 x 2048 -> 2048 4.9
//   [8.3]), or of 12 KB and 13 MB (16 x 6144 -> 1000 6.4 [10.9]); f32, whose MFMAs
//   are 16 times slower, of 16 KB and 17 MB (16 x 2048 -> 2048 6.5 [9.1], 32 x 4096
//   -> 1024 9.8 [12.7]);
//   up to 64: rows of 8 KB, 13 MB in all (64 x 4096 -> 1024 f16 5.4 [8.6], f32 64 x
//   1536 -> 2048 7.6 [8.3]; but f32 64 x 1024 -> 4096 9.9 [9.4]);
//   above: 64 rows per block; 16-column blocks where they fit one round of the
//   256 CUs, f16 to rows of 6 KB (128 x 2048 -> 1000 6.3 [7.4], 100 x 2048 -> 64 5.5
//   [7.3], 100 x 3072 -> 200 7.8 [7.3]; but 128 x 4096 -> 512 9.0 [7.5]), 4 KB where
//   they are no whole vectors (128 x 3002 -> 200 10.7 [8.7]), beyond 512 input rows
//   of 3 KB (1000 x 1536 -> 200 7.1 [7.2]; but 1000 x 2048 -> 200 8.3 [7.6], 1000 x
//   3072 -> 200 11.1 [9.2]), f32 of 2.5 KB (200 x 576 -> 1000 6.9 [7.5]; but 128 x 770
//   -> 200 8.2 [7.2], 256 x 1024 -> 200 8.9 [7.2]);
//   f16 32-column blocks that are no more than 256 and read up to 1 M bytes of k
//   together (512 x 2048 -> 1000 8.2 [9.1], 400 x 752 -> 1536 8.0 [8.4]), or no more
//   than 512 with rows of 1.6 KB (1000 x 576 -> 1000 6.8 [7.5], 512 x 770 -> 2048 8.8
//   [8.4]; but 200 x 1024 -> 4096 8.9 [8.2]).
template <typename T>
hipError_t skinny(const T *x, const T *w, const T *bias, T *y, size_t rows, size_t in, size_t out,
                  hipStream_t s) {
    constexpr bool f32 = sizeof(T) == 4;
    const size_t row = in * sizeof(T);
    if (row < 16 || row > 16384 || out > (size_t{1} << 24)) return hipErrorNotSupported;
    const size_t total = row * out, tiles = (out + 15) / 16, groups = (rows + 15) / 16;
    if (rows > 64) {
        if (rows > (size_t{1} << 20)) return hipErrorNotSupported;
        const size_t narrow = tiles * ((rows + 63) / 64), wide = (tiles + 1) / 2 * ((rows + 63) / 64);
        if (narrow <= 256 && row <= (f32 ? 2560u : rows > 512 ? 3072u : row % 16 == 0 ? 6144u : 4096u))
            return launch_skinny<T, 4, 1, 8, 1>(x, w, bias, y, rows, in, out, s);
        if constexpr (!f32)
            if (row <= (rows <= 512 ? 4096u : 3072u) && (wide <= 256 ? wide * row <= (1u << 20) : wide <= 512 && row <= 1600))
                return launch_skinny<T, 4, 2, 4, 1>(x, w, bias, y, rows, in, out, s);
        return hipErrorNotSupported;
    }
    const bool few = rows <= 32;
    const bool small = f32 ? (few ? total <= (17u << 20) && row <= 16384u : total <= (13u << 20) && row <= 8192u)
                           : (total <= (34u << 20) && row <= 8192u && few) ||
                                 (total <= (13u << 20) && row <= (few ? 12288u : 8192u));
    if (!small) return hipErrorNotSupported;
    // One 16-row group per block where all groups' blocks fit the 256 CUs
    // (the weights again from L2: 32 x 4096 -> 1024 f16 5.4 us, two groups 6.7)
    // or there is only one; else two. From a second round of 16-column blocks
    // on, 32 columns (32 x 1024 -> 16384 9.2, 16 columns 11.1).
    if (tiles > 256) return launch_skinny<T, 2, 2, 8, 1>(x, w, bias, y, rows, in, out, s);
    if (groups == 1 || tiles * groups <= 256) return launch_skinny<T, 1, 1, 8, 2>(x, w, bias, y, rows, in, out, s);
    return launch_skinny<T, 2, 1, 8, 1>(x, w, bias, y, rows, in, out, s);
}

}  // namespace

hipError_t linear_small(bool f32, const void *x, const void *w, const void *bias, void *y,
                        size_t rows, size_t in, size_t out, hipStream_t s) {
    const size_t elem = f32 ? 4 : 2;
    if (rows == 0 || in == 0 || out == 0) return hipErrorNotSupported;
    // The GEMV launch is one wave (64 work-items) per output row: out * 64 must
    // stay below 2^32, the dispatch packet's work-item count. A larger `out`
    // is declined here (hipErrorNotSupported), and the caller takes the
    // library GEMM.
    const bool stream = rows <= kGemvMaxRows && in % (16 / elem) == 0 && in <= 0xffffffffu &&
                        out <= 0xffffffffu / kWave && (((uintptr_t)x | (uintptr_t)w) & 15u) == 0;
    if (f32) {
        const float *fx = static_cast<const float *>(x), *fw = static_cast<const float *>(w);
        const float *fb = static_cast<const float *>(bias);
        return stream ? gemv(fx, fw, fb, static_cast<float *>(y), rows, in, out, s)
                      : skinny(fx, fw, fb, static_cast<float *>(y), rows, in, out, s);
    }
    const _Float16 *hx = static_cast<const _Float16 *>(x), *hw = static_cast<const _Float16 *>(w);
    const _Float16 *hb = static_cast<const _Float16 *>(bias);
    return stream ? gemv(hx, hw, hb, static_cast<_Float16 *>(y), rows, in, out, s)
                  : skinny(hx, hw, hb, static_cast<_Float16 *>(y), rows, in, out, s);
}

}  // namespace k
}  // namespace icsdk
