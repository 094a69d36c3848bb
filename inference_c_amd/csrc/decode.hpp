// Attention of few query rows (k_attention_decode.hip): plan and launch.
#pragma once

#include "flash.hpp"

namespace icsdk {
namespace flash {

struct DecodePlan {
    bool use = false;
    uint32_t row_groups = 1;  // groups of 16 packed rows, a block each
    uint32_t parts = 1;       // parts of the key range, a block each
};
struct DecodeArgs {
    uint32_t parts, row_groups;
};

// `use` is false where the flash or row kernels serve the call.
DecodePlan decode_plan(const k::SdpaShape &sh, bool aligned, bool f32, bool causal);
// Bytes of the parts' results, 0 for one part.
size_t decode_workspace(const DecodePlan &p, const k::SdpaShape &sh);
// a: shape, scale and causal fields, part_o and part_ml for several parts.
hipError_t launch_decode_f16(const DecodePlan &p, const _Float16 *q, const _Float16 *k, const _Float16 *v,
                             const _Float16 *mask, _Float16 *out, const SdpaArgs &a, hipStream_t s);
hipError_t launch_decode_f32(const DecodePlan &p, const float *q, const float *k, const float *v,
                             const float *mask, float *out, const SdpaArgs &a, hipStream_t s);

}  // namespace flash
}  // namespace icsdk
