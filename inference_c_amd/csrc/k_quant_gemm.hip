// Quantized linear of many input rows (prompts): y[r][o] = f16(sum_b scale_b *
// sum_k x[r][32 b + k] q_bk) for Q8_0 and Q4_0 weights, as a tiled matrix
// product.
//
// A block of four waves owns 32 MT rows of x and 128 output columns; a wave
// takes all the rows and 32 columns, so every weight is decoded once per
// block and by one lane. Steps of two 32-weight blocks: x as [row][k] f16 and
// the packed values as [column][block] bytes are double-buffered in LDS, the
// next step's loads in flight while the current one is computed. The values
// of a block start 2 bytes after its f16 scale, at any even address: they are
// loaded as 16 bytes from there as they are (gfx950 serves unaligned vectors)
// and lie aligned in LDS.
//
// v_mfma_f32_32x32x16_f16, A = x (lane l: row l % 32), B = weights (lane l:
// column l % 32), two per block of 32 weights. The sum over k may run in any
// order as long as x and the weights agree: Q8 lane half h = l / 32 takes
// weights 16 h + 8 j .. + 7 in MFMA j (its 16 bytes of the block), Q4 weights
// 16 j + 8 h .. + 7 (low and high nibbles of its 8 bytes). A value byte
// (Q8: q + 128 after an XOR; Q4: n) spreads to the f16 subnormal u 2^-24 by
// v_perm_b32, and one packed subtraction removes the offset, leaving q 2^-24
// exactly. D holds one block's products for 16 rows of the lane's column, so
// one scale per lane multiplies them into the f32 accumulators (the scale
// never meets f16); 2^24 comes back at the end.
//
// Bound: per wave and block MT * 64 cycles of MFMA and about as many of VALU
// (16 MT scale FMAs, 20 of decode), which overlap only between the two waves
// of a SIMD, and the LDS reads (9 KB per wave and block at MT 4). Measured
// (us, weights decoded again for every 16 rows before -> here): Q8_0 512 x 4096
// -> 14336 400 -> 101 (593 TFLOP/s), 2048 x 4096 -> 4096 400 -> 109, Q4_0 303 ->
// 97 and 300 -> 102. Reading ahead inside a step by hand (a chain of MFMA
// pairs, each scaled under the next) took 256 registers and 154 us.
#include "kern_common.hpp"
#include "kernels.hpp"
#include "quant_common.hpp"

namespace icsdk {
namespace k {
namespace {

typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_2 __attribute__((ext_vector_type(4), aligned(2)));

constexpr uint32_t kCols = 128;        // output columns per block
constexpr uint32_t kStepBlocks = 2;    // 32-weight blocks per step
constexpr uint32_t kXPitch = kStepBlocks * 64 + 16;   // LDS bytes per x row

template <bool kQ8, int MT>
__global__ __launch_bounds__(kBlock) void quant_gemm_kernel(const uint16_t *__restrict__ x,
                                                            const uint8_t *__restrict__ w,
                                                            uint16_t *__restrict__ y, uint32_t rows,
                                                            uint32_t in, uint32_t out,
                                                            uint32_t row_blocks) {
    constexpr uint32_t kBytes = Fmt<kQ8>::kBytes;
    constexpr uint32_t kRows = 32 * MT;
    constexpr uint32_t kValues = kBytes - 2;                     // value bytes of a block: 32 or 16
    constexpr uint32_t kWPitch = kStepBlocks * kValues + 16;     // LDS bytes per column
    constexpr uint32_t kXVecs = kRows * kStepBlocks * 4 / kBlock; // 16-byte vectors per thread and step
    constexpr uint32_t kWVecs = kCols * kStepBlocks * (kValues / 16) / kBlock;
    static_assert(kXVecs * kBlock == kRows * kStepBlocks * 4 && kWVecs * kBlock == kCols * kStepBlocks * kValues / 16,
                  "whole vectors per thread");
    static_assert(kCols * kStepBlocks == kBlock, "one scale per thread");
    __shared__ __attribute__((aligned(16))) uint8_t xs[2][kRows * kXPitch];
    __shared__ __attribute__((aligned(16))) uint8_t ws[2][kCols * kWPitch];
    __shared__ float ss[2][kStepBlocks][kCols];
    const uint32_t tid = threadIdx.x, lane = tid & 63, col = lane & 31, half = lane >> 5;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid / kWave);
    // Blocks go round-robin over the 8 XCDs: the row blocks of one column
    // block are neighbours on one XCD, whose L2 then serves its weights again
    const uint32_t xcd = blockIdx.x % 8, seq = blockIdx.x / 8;
    const uint32_t col_block = seq / row_blocks * 8 + xcd, row_block = seq % row_blocks;
    const uint32_t o_first = col_block * kCols, r_first = row_block * kRows;
    if (o_first >= out) return;
    const uint32_t blocks = in / 32;
    const uint64_t row_bytes = (uint64_t)blocks * kBytes;

    // Loads of a step (blocks b0, b0 + 1): rows, columns and blocks past the
    // end are clamped onto the last one (not stored; a block past the end gets
    // scale 0 when stashed: its products count 0, or make a sum that x's
    // infinities or NaN leave not finite anyway NaN, which is then redone).
    struct Stage {
        u32x4 x[kXVecs], w[kWVecs];
        uint16_t scale;
    };
    auto fetch = [&](Stage &g, uint32_t b0) {
#pragma unroll
        for (uint32_t i = 0; i < kXVecs; ++i) {
            const uint32_t e = tid + kBlock * i, r = min(r_first + e / (kStepBlocks * 4), rows - 1);
            const uint32_t k = min(b0 * 32 + e % (kStepBlocks * 4) * 8, in - 8);
            g.x[i] = *reinterpret_cast<const u32x4 *>(x + (uint64_t)r * in + k);
        }
#pragma unroll
        for (uint32_t i = 0; i < kWVecs; ++i) {
            constexpr uint32_t kPer = kStepBlocks * kValues / 16;   // vectors per column
            const uint32_t e = tid + kBlock * i, o = min(o_first + e / kPer, out - 1), v = e % kPer;
            const uint32_t b = min(b0 + v / (kValues / 16), blocks - 1);
            g.w[i] = *reinterpret_cast<const u32x4_2 *>(w + o * row_bytes + (uint64_t)b * kBytes + 2 +
                                                       v % (kValues / 16) * 16);
        }
        const uint32_t o = min(o_first + tid / kStepBlocks, out - 1), b = min(b0 + tid % kStepBlocks, blocks - 1);
        g.scale = *reinterpret_cast<const uint16_t *>(w + o * row_bytes + (uint64_t)b * kBytes);
    };
    auto stash = [&](const Stage &g, uint32_t buf, uint32_t b0) {
#pragma unroll
        for (uint32_t i = 0; i < kXVecs; ++i) {
            const uint32_t e = tid + kBlock * i;
            *reinterpret_cast<u32x4 *>(&xs[buf][e / (kStepBlocks * 4) * kXPitch + e % (kStepBlocks * 4) * 16]) = g.x[i];
        }
#pragma unroll
        for (uint32_t i = 0; i < kWVecs; ++i) {
            constexpr uint32_t kPer = kStepBlocks * kValues / 16;
            const uint32_t e = tid + kBlock * i;
            *reinterpret_cast<u32x4 *>(&ws[buf][e / kPer * kWPitch + e % kPer * 16]) = g.w[i];
        }
        ss[buf][tid % kStepBlocks][tid / kStepBlocks] =
            b0 + tid % kStepBlocks < blocks ? (float)__builtin_bit_cast(_Float16, g.scale) : 0.0f;
    };

    float16v acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.0f;
    const uint8_t *xbase = &xs[0][0] + col * kXPitch + (kQ8 ? 32 : 16) * half;
    const uint8_t *wbase = &ws[0][0] + (32 * wave + col) * kWPitch + (kQ8 ? 16 : 8) * half;

    auto compute = [&](uint32_t buf) {
        const uint8_t *xb = xbase + buf * sizeof(xs[0]), *wb = wbase + buf * sizeof(ws[0]);
#pragma unroll
        for (uint32_t s = 0; s < kStepBlocks; ++s) {
            const float scale = ss[buf][s][32 * wave + col];
            half8 bf[2];
            if constexpr (kQ8) {
                const u32x4 u = *reinterpret_cast<const u32x4 *>(wb + s * kValues) ^ 0x80808080u;
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    bf[j] = spread_values(u[2 * j], u[2 * j + 1], 0x80808080u);
            } else {
                const u32x2 u = *reinterpret_cast<const u32x2 *>(wb + s * kValues);
                bf[0] = spread_values(u.x & 0x0f0f0f0fu, u.y & 0x0f0f0f0fu, 0x80088008u);
                bf[1] = spread_values(u.x >> 4 & 0x0f0f0f0fu, u.y >> 4 & 0x0f0f0f0fu, 0x80088008u);
            }
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const uint8_t *xa = xb + 32 * t * kXPitch + s * 64;
                const half8 a0 = *reinterpret_cast<const half8 *>(xa);
                const half8 a1 = *reinterpret_cast<const half8 *>(xa + (kQ8 ? 16 : 32));
                float16v d;
#pragma unroll
                for (int r = 0; r < 16; ++r) d[r] = 0.0f;
                d = __builtin_amdgcn_mfma_f32_32x32x16_f16(a0, bf[0], d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_32x32x16_f16(a1, bf[1], d, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[t][r] = __builtin_fmaf(scale, d[r], acc[t][r]);
            }
        }
    };

    // Two steps of loads in flight: step s computes from LDS buffer s % 2 while
    // step s + 1 waits in one register stage and step s + 2 is loading into the
    // other. (Loads past the end repeat the last block; not used.)
    Stage stage[2];
    fetch(stage[0], 0);
    fetch(stage[1], kStepBlocks);
    stash(stage[0], 0, 0);
    fetch(stage[0], 2 * kStepBlocks);
    __syncthreads();
    for (uint32_t b0 = 0; b0 < blocks; b0 += 2 * kStepBlocks) {
        compute(0);
        stash(stage[1], 1, b0 + kStepBlocks);
        fetch(stage[1], b0 + 3 * kStepBlocks);
        __syncthreads();
        if (b0 + kStepBlocks >= blocks) break;
        compute(1);
        stash(stage[0], 0, b0 + 2 * kStepBlocks);
        fetch(stage[0], b0 + 4 * kStepBlocks);
        __syncthreads();
    }
    const uint32_t o = o_first + 32 * wave + col;
    if (o >= out) return;
    uint64_t bad = 0;   // outputs whose sum is not finite
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const uint32_t row = r_first + 32 * t + 8 * (r / 4) + 4 * half + r % 4;
            const float v = acc[t][r] * 0x1p24f;
            if (row < rows) {
                y[(uint64_t)row * out + o] = __builtin_bit_cast(uint16_t, (_Float16)v);
                if (!__builtin_isfinite(v)) bad |= uint64_t{1} << (16 * t + r);
            }
        }
    // rare (an x row holding an infinity or NaN): the reference's chain, one
    // output at a time
#pragma unroll 1
    while (bad != 0) {
        const uint32_t i = (uint32_t)__builtin_ctzll(bad), r = i % 16;
        bad &= bad - 1;
        const uint32_t row = r_first + 32 * (i / 16) + 8 * (r / 4) + 4 * half + r % 4;
        const float v = reference_chain<kQ8>(x + (uint64_t)row * in, w + o * row_bytes, blocks);
        y[(uint64_t)row * out + o] = __builtin_bit_cast(uint16_t, (_Float16)v);
    }
}

template <bool kQ8>
hipError_t gemm(const uint16_t *x, const uint8_t *w, uint16_t *y, size_t rows, size_t in, size_t out,
                int mt, hipStream_t s) {
    const size_t row_blocks = (rows + 32 * mt - 1) / (32 * mt);
    const size_t col_blocks = (out + kCols - 1) / kCols;
    const size_t grid = (col_blocks + 7) / 8 * 8 * row_blocks;
    if (grid > 0xffffff) return hipErrorNotSupported;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kBlock), 0, s, x, w, y, (uint32_t)rows,
                           (uint32_t)in, (uint32_t)out, (uint32_t)row_blocks);
        return hipGetLastError();
    };
    if (mt == 1) return go(quant_gemm_kernel<kQ8, 1>);
    if (mt == 2) return go(quant_gemm_kernel<kQ8, 2>);
    return go(quant_gemm_kernel<kQ8, 4>);
}

}  // namespace

hipError_t quant_gemm(bool q8, const uint16_t *x, const uint8_t *w, uint16_t *y, size_t rows, size_t in,
                      size_t out, hipStream_t s) {
    if (rows > 0x7fffffffu || out > 0x7fffffffu || in > 0x7fffffffu) return hipErrorNotSupported;
    // Rows per block by a model of the measured times: a step (64 k) of a
    // block alone on its CU takes `chain` us, several on a CU `shared` us each;
    // quant_mma_kernel (16 rows x 64 columns per block) takes `mma_chain` us per
    // 4096 k alone and `mma_shared` per 256 blocks. It stays the faster one
    // where the tiles here leave most CUs without a block. Fitted to 17 shapes
    // of 17 .. 2048 rows per format, [576 .. 14336, 777 .. 14336]; e.g. Q8_0 us,
    // mma / 32 / 64 / 128 rows: 64 x 4096 -> 4096 19.6 / 35 / 51 / 67, 256 x 4096
    // -> 4096 52 / 38 / 52 / 68, 512 x 4096 -> 14336 400 / 202 / 131 / 101.
    struct Cost {
        double chain[3], shared[3], mma_chain, mma_shared;
    };
    static constexpr Cost kQ8Cost = {{0.55, 0.79, 1.05}, {0.45, 0.55, 0.82}, 18.7, 14.0};
    static constexpr Cost kQ4Cost = {{0.45, 0.66, 1.11}, {0.40, 0.49, 0.78}, 13.7, 10.7};
    const Cost &c = q8 ? kQ8Cost : kQ4Cost;
    const double steps = (double)in / 64;
    const double mma_rounds = (double)((rows + 15) / 16) * (double)((out + 63) / 64) / 256;
    double best = (double)in / 4096 * (mma_rounds * c.mma_shared > c.mma_chain ? mma_rounds * c.mma_shared : c.mma_chain);
    int mt = 0;
    for (int i = 0; i < 3; ++i) {
        const size_t blocks = (rows + (32u << i) - 1) / (32u << i) * ((out + kCols - 1) / kCols);
        const double shared = (double)((blocks + 255) / 256) * c.shared[i];
        const double us = steps * (shared > c.chain[i] ? shared : c.chain[i]);
        if (us < (mt == 0 ? 0.92 : 1.0) * best) {   // (the model is good to a few percent)
            best = us;
            mt = 1 << i;
        }
    }
    if (mt == 0) return hipErrorNotSupported;
    return q8 ? gemm<true>(x, w, y, rows, in, out, mt, s) : gemm<false>(x, w, y, rows, in, out, mt, s);
}

}  // namespace k
}  // namespace icsdk
