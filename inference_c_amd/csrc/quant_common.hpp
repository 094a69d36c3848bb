// What the quantized-linear kernels share (k_quant.hip, k_quant_gemm.hip): the
// packed formats, their value decoding and the reference's own chain.
#pragma once

#include "kern_common.hpp"

namespace icsdk {
namespace k {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));

template <bool kQ8> struct Fmt {
    static constexpr uint32_t kBytes = kQ8 ? 34 : 18;
};

__device__ inline half2_t as_half2(uint32_t bits) { return __builtin_bit_cast(half2_t, bits); }

// Eight value bytes u (four per word) as f16 (u + offset) 2^-24, exact:
// v_perm_b32 spreads two bytes to the halves 0x00uu (subnormals) and the
// packed addition of `offset` (a pair of subnormals of that unit) is exact.
__device__ inline half8 spread_values(uint32_t lo, uint32_t hi, uint32_t offset) {
    const half2_t add = as_half2(offset);
    const half2_t p[4] = {as_half2(__builtin_amdgcn_perm(0u, lo, 0x0c010c00u)) + add,
                          as_half2(__builtin_amdgcn_perm(0u, lo, 0x0c030c02u)) + add,
                          as_half2(__builtin_amdgcn_perm(0u, hi, 0x0c010c00u)) + add,
                          as_half2(__builtin_amdgcn_perm(0u, hi, 0x0c030c02u)) + add};
    return half8{p[0].x, p[0].y, p[1].x, p[1].y, p[2].x, p[2].y, p[3].x, p[3].y};
}

// One output by the reference's own chain (tensor_compute_cuda.cu:216-238):
// sum = fmaf(x_k, scale_b * q_k, sum) over the blocks b of the row, then the
// 32 values k of each, from 0. The fix-up for an output whose fast sum is
// not finite. Finite x and finite scales keep every partial sum of the fast
// kernels finite (at most ~2^30 for f16 operands), and a non-finite x makes
// the reference's sum non-finite too, but the offset decode forms
// x (q + offset) - offset x, so x = +-Inf gives Inf - Inf = NaN where the
// reference's x * (scale q) gives +-Inf (NaN only for q = 0, a zero scale
// or infinities of both signs). Running the reference's chain for those
// outputs makes them equal to the reference's bit for bit. `xrow` is the
// input row (16-byte aligned), `wrow` the packed weight row (2-byte
// aligned). Rare: only rows with an infinity or NaN take it.
template <bool kQ8>
__device__ inline float reference_chain(const uint16_t *xrow, const uint8_t *wrow,
                                        uint32_t blocks) {
    constexpr uint32_t kBytes = Fmt<kQ8>::kBytes;
    float sum = 0.0f;
#pragma unroll 1
    for (uint32_t b = 0; b < blocks; ++b) {
        const uint16_t *blk = reinterpret_cast<const uint16_t *>(wrow + (uint64_t)b * kBytes);
        uint16_t half_words[kBytes / 2];
#pragma unroll
        for (uint32_t i = 0; i < kBytes / 2; ++i) half_words[i] = blk[i];
        const u32x4 *xp = reinterpret_cast<const u32x4 *>(xrow + (uint64_t)b * 32);
        uint32_t xw[16];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const u32x4 t = xp[v];
            xw[4 * v] = t.x;
            xw[4 * v + 1] = t.y;
            xw[4 * v + 2] = t.z;
            xw[4 * v + 3] = t.w;
        }
        const float scale = (float)__builtin_bit_cast(_Float16, half_words[0]);
#pragma unroll
        for (uint32_t k = 0; k < 32; ++k) {
            int q;
            if constexpr (kQ8) {
                const uint32_t byte = k;   // value byte k sits at block byte 2 + k
                q = (int)(int8_t)(uint8_t)(half_words[1 + byte / 2] >> (8 * (byte & 1)));
            } else {
                const uint32_t byte = k & 15;
                const uint8_t packed = (uint8_t)(half_words[1 + byte / 2] >> (8 * (byte & 1)));
                q = (int)(k < 16 ? packed & 15 : packed >> 4) - 8;
            }
            const uint16_t xb = (uint16_t)(xw[k / 2] >> (16 * (k & 1)));
            sum = __builtin_fmaf((float)__builtin_bit_cast(_Float16, xb), scale * (float)q, sum);
        }
    }
    return sum;
}

// Matrix form for many rows (k_quant_gemm.hip): hipErrorNotSupported for what
// it does not take. x rows 16-byte aligned, w 4-byte aligned.
hipError_t quant_gemm(bool q8, const uint16_t *x, const uint8_t *w, uint16_t *y, size_t rows, size_t in,
                      size_t out, hipStream_t s);

}  // namespace k
}  // namespace icsdk
