// Row operations for rows of any width and element alignment (k_rowany.hip):
// narrow rows, rows that are not whole 16-byte vectors, and rows too long for
// one block's registers. Each returns hipErrorNotSupported for what it does
// not take (rows of less than one vector; rows of more than 4096 vectors
// without scratch memory or under stream capture).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace icsdk {
namespace row_any {

// Rows of at most this many 16-byte vectors run fastest here also when they
// are whole aligned vectors: several rows share a wave.
constexpr size_t kNarrowVectors = 32;

template <typename S>
hipError_t rms_norm(const S *x, const S *residual, S *sum_out, const S *w, S *y, size_t rows,
                    size_t width, float eps, hipStream_t s);
template <typename S>
hipError_t layer_norm(const S *x, const S *scale, const S *bias, S *y, size_t rows, size_t width,
                      float eps, hipStream_t s);
template <typename S>
hipError_t softmax(const S *x, S *y, size_t rows, size_t width, size_t q_len,
                   size_t causal_offset, hipStream_t s);
template <typename S, bool kMax>
hipError_t reduce(const S *x, float *y, size_t rows, size_t width, hipStream_t s);

}  // namespace row_any
}  // namespace icsdk
