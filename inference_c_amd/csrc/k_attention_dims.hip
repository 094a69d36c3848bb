// Flash attention for head dims other than 64 and 128: the kernels of
// flash.hpp compiled for padded dims, with the rows' true widths as arguments.
// f16 P is carried as an f16 pair (hi + lo), so it keeps the f32 accuracy of
// the row kernel that served these dims before; that doubles the P V MFMAs.
// Rows whose output is not finite although their sum is (an infinite value)
// are done again by the row routine at the kernel's end.
// Measured (us, row kernel -> here): f16 16 heads x 1025^2 D 80 1711 -> 24.7,
// 16 x 1024^2 D 96 2209 -> 28.7, 8 x 1024^2 D 256 causal 1713 -> 78 (16
// heads), f32 16 x 1025^2 D 80 ~2000 -> 104. Bound like the D 64 / 128
// kernels: MFMA, softmax VALU and LDS phases that overlap only partly.
#include "flash.hpp"

namespace icsdk {
namespace flash {
namespace {

// One launch of the (mask, split) form of a (D, BM, KS) kernel.
#define ICSDK_ANY_DIM(KERNEL, D, BM, KS)                                                       \
    do {                                                                                       \
        if (variant.general && variant.split)                                                  \
            hipLaunchKernelGGL((KERNEL<D, BM, true, true, KS, true>), grid, block, 0, s, q, k, \
                               v, mask, out, a);                                               \
        else if (variant.general)                                                              \
            hipLaunchKernelGGL((KERNEL<D, BM, true, false, KS, true>), grid, block, 0, s, q,   \
                               k, v, mask, out, a);                                            \
        else if (variant.split)                                                                \
            hipLaunchKernelGGL((KERNEL<D, BM, false, true, KS, true>), grid, block, 0, s, q,   \
                               k, v, mask, out, a);                                            \
        else                                                                                   \
            hipLaunchKernelGGL((KERNEL<D, BM, false, false, KS, true>), grid, block, 0, s, q,  \
                               k, v, mask, out, a);                                            \
        return hipGetLastError();                                                              \
    } while (0)

template <int D>
hipError_t launch_f16(const FlashVariant &variant, dim3 grid, dim3 block, hipStream_t s,
                      const _Float16 *q, const _Float16 *k, const _Float16 *v,
                      const _Float16 *mask, _Float16 *out, const SdpaArgs &a) {
    if constexpr (D <= 128) {
        if (variant.key_parts == 2) {
            if (variant.bm == 64) ICSDK_ANY_DIM(sdpa_flash_kernel, D, 64, 2);
            ICSDK_ANY_DIM(sdpa_flash_kernel, D, 128, 2);
        }
        if (variant.bm == 256) ICSDK_ANY_DIM(sdpa_flash_kernel, D, 256, 1);
    }
    if (variant.bm == 128) ICSDK_ANY_DIM(sdpa_flash_kernel, D, 128, 1);
    ICSDK_ANY_DIM(sdpa_flash_kernel, D, 64, 1);
}

template <int D>
hipError_t launch_f32(const FlashVariant &variant, dim3 grid, dim3 block, hipStream_t s,
                      const float *q, const float *k, const float *v, const float *mask,
                      float *out, const SdpaArgs &a) {
    if (variant.bm == 128) ICSDK_ANY_DIM(sdpa_flash_f32_kernel, D, 128, 1);
    ICSDK_ANY_DIM(sdpa_flash_f32_kernel, D, 64, 1);
}

#undef ICSDK_ANY_DIM

}  // namespace

hipError_t launch_any_dim_f16(const FlashVariant &variant, dim3 grid, dim3 block, hipStream_t s,
                              const _Float16 *q, const _Float16 *k, const _Float16 *v,
                              const _Float16 *mask, _Float16 *out, const SdpaArgs &a) {
    switch (variant.dim) {
    case 32: return launch_f16<32>(variant, grid, block, s, q, k, v, mask, out, a);
    case 80: return launch_f16<80>(variant, grid, block, s, q, k, v, mask, out, a);
    case 96: return launch_f16<96>(variant, grid, block, s, q, k, v, mask, out, a);
    case 128: return launch_f16<128>(variant, grid, block, s, q, k, v, mask, out, a);
    case 256: return launch_f16<256>(variant, grid, block, s, q, k, v, mask, out, a);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_any_dim_f32(const FlashVariant &variant, dim3 grid, dim3 block, hipStream_t s,
                              const float *q, const float *k, const float *v, const float *mask,
                              float *out, const SdpaArgs &a) {
    switch (variant.dim) {
    case 32: return launch_f32<32>(variant, grid, block, s, q, k, v, mask, out, a);
    case 80: return launch_f32<80>(variant, grid, block, s, q, k, v, mask, out, a);
    case 96: return launch_f32<96>(variant, grid, block, s, q, k, v, mask, out, a);
    case 128: return launch_f32<128>(variant, grid, block, s, q, k, v, mask, out, a);
    case 256: return launch_f32<256>(variant, grid, block, s, q, k, v, mask, out, a);
    default: return hipErrorInvalidValue;
    }
}

}  // namespace flash
}  // namespace icsdk
