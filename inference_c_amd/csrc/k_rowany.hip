// Row operations for rows of any width and element alignment: RMSNorm (with
// and without the residual add), LayerNorm, softmax, row sum and row max.
//
// A group of T lanes owns a row and holds it in registers, NV vectors per
// lane. A row need not be whole 16-byte vectors: its last vector is the row's
// last 16 bytes, so it overlaps the one before; the overlap counts once in
// the reductions, and both lanes store the same values there. Loads and
// stores are 16 bytes at any element alignment (gfx950 serves them as they
// are; a 64-lane access then touches 9 lines instead of 8).
//   T 8, 16, 32   several rows per wave, for rows of at most 32 vectors
//   T 64          a wave per row
//   T 256, 1024   a block per row, partial results through LDS
// Rows of more than 4096 vectors are cut into parts over several blocks (f32 rows
// of up to 8192 only where there are fewer than 128 of them): a first launch
// leaves each part's partial result, a second folds a row's partials and writes
// the output, reading its part again (from L2 where it fits).
//
// Bound: HBM bytes (one read, one write; the split form reads twice, the
// second time mostly from cache); below about 8 MB the launches.
// Measured (us, scalar one-block-per-row kernel or one wave per narrow row ->
// here): softmax f32 [32, 128256] 380 -> 13.9, [1, 28289] 65 -> 9.6, f16
// [4, 23568] 50 -> 4.8, [200000, 64] 43 -> 10.0; LayerNorm f32 [149, 94705]
// 413 -> 32.5; RMSNorm f16 [6880, 965] 10.3 -> 5.9; row sum f16 [41505, 71]
// 10.7 -> 4.3.
#include "kern_common.hpp"
#include "row_any.hpp"
#include "sdk.hpp"

namespace icsdk {
namespace row_any {
namespace {

typedef uint32_t u32x4_2 __attribute__((ext_vector_type(4), aligned(2)));

template <typename S> __device__ inline Vec16<S> load_any(const S *p) {
    const u32x4_2 raw = __builtin_nontemporal_load(reinterpret_cast<const u32x4_2 *>(p));
    return __builtin_bit_cast(Vec16<S>, raw);
}
template <typename S> __device__ inline Vec16<S> load_param(const S *p) {
    const u32x4_2 raw = *reinterpret_cast<const u32x4_2 *>(p);
    return __builtin_bit_cast(Vec16<S>, raw);
}
template <typename S> __device__ inline void store_any(S *p, const Vec16<S> &v) {
    __builtin_nontemporal_store(__builtin_bit_cast(u32x4_2, v), reinterpret_cast<u32x4_2 *>(p));
}

// ---- reductions over a row's T lanes; every lane gets the result ---------------

template <int T> constexpr int lds_floats() { return T > kWave ? T / kWave : 1; }

template <int T, bool kMax> __device__ inline float row_fold(float v, float *lds) {
    auto op = [](float a, float b) { return kMax ? fmaxf(a, b) : a + b; };
    if constexpr (T < kWave) {
        // the lanes of a DPP row all hold values: no lane is left out
        v = op(v, dpp_f32<kQuadSwap1>(v, v));
        v = op(v, dpp_f32<kQuadSwap2>(v, v));
        v = op(v, dpp_f32<kRowHalfMirror>(v, v));
        if constexpr (T >= 16) v = op(v, dpp_f32<kRowMirror>(v, v));
        if constexpr (T >= 32) v = op(v, __shfl_xor(v, 16, kWave));
        return v;
    } else {
        v = kMax ? wave_max(v) : wave_sum(v);
        if constexpr (T > kWave) {
            const uint32_t wave = threadIdx.x / kWave;
            __syncthreads();
            if (threadIdx.x % kWave == 0) lds[wave] = v;
            __syncthreads();
            v = lds[0];
#pragma unroll
            for (int i = 1; i < T / kWave; ++i) v = op(v, lds[i]);
        }
        return v;
    }
}
template <int T> __device__ inline float row_total(float v, float *lds) { return row_fold<T, false>(v, lds); }
template <int T> __device__ inline float row_largest(float v, float *lds) { return row_fold<T, true>(v, lds); }

// ---- a lane's share of a row (or of a part of a row) ----------------------------

// Vectors first .. end - 1 of a row of `width` elements; lane t holds vectors
// first + t, first + t + T, ... . Vector vi starts at element at(j): E vi, or
// the row's last E elements for a last partial vector.
template <typename S, int T, int NV> struct Share {
    static constexpr int E = Vec16<S>::N;
    Vec16<S> v[NV];
    uint32_t start[NV], lead[NV];   // first element; elements of it another lane counts (E: all)

    __device__ inline void place(uint32_t t, uint32_t width, uint32_t first, uint32_t end) {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const uint32_t vi = first + t + j * T;
            start[j] = min(vi * (uint32_t)E, width - E);
            lead[j] = vi < end ? vi * (uint32_t)E - start[j] : (uint32_t)E;
        }
    }
    __device__ inline void load(const S *row) {
#pragma unroll
        for (int j = 0; j < NV; ++j) v[j] = load_any(row + start[j]);
    }
    __device__ inline bool any(int j) const { return lead[j] < (uint32_t)E; }
    __device__ inline bool counts(int j, int e) const { return (uint32_t)e >= lead[j]; }
    __device__ inline float at(int j, int e) const { return Elem<S>::load(v[j].v[e]); }
    __device__ inline void params(const S *p, Vec16<S> (&out)[NV]) const {
#pragma unroll
        for (int j = 0; j < NV; ++j) out[j] = load_param(p + start[j]);
    }
    // out(j, e) for every vector of the lane
    template <typename F> __device__ inline void store(S *row, bool live, F &&out) const {
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            Vec16<S> o;
#pragma unroll
            for (int e = 0; e < E; ++e) o.v[e] = Elem<S>::store(out(j, e));
            if (live && any(j)) store_any(row + start[j], o);
        }
    }
};

// The row and lane of a thread; rows past the end are clamped onto the last
// one (computed, not stored).
template <int T> struct Slot {
    size_t row;
    uint32_t t;
    bool live;
    __device__ explicit Slot(size_t rows) {
        size_t r;
        if constexpr (T > kWave) {
            r = blockIdx.x;
            t = threadIdx.x;
        } else {
            r = (size_t)blockIdx.x * (kBlock / T) + threadIdx.x / T;
            t = threadIdx.x % T;
        }
        live = r < rows;
        row = live ? r : rows - 1;
    }
};

template <int T> constexpr int block_threads() { return T > kBlock ? T : kBlock; }

template <typename S> __device__ inline float num_exp(float x) {
    if constexpr (sizeof(S) == 2) return fast_exp(x);
    else return expf(x);
}

// Visible keys of a causal row: 0 .. limit.
__device__ inline uint32_t causal_limit(size_t row, uint32_t width, size_t q_len, size_t offset) {
    if (q_len == 0) return width;
    const uint64_t limit = (uint64_t)(row % q_len) + offset;
    return (uint32_t)(limit < width ? limit : width);
}

// ---- one group per row -------------------------------------------------------------

template <typename S, int T, int NV, bool kResidual>
__global__ __launch_bounds__(block_threads<T>()) void rms_kernel(const S *x, const S *residual,
                                                                 S *sum_out, const S *w, S *y,
                                                                 size_t rows, uint32_t width,
                                                                 float eps) {
    __shared__ float lds[lds_floats<T>()];
    constexpr int E = Vec16<S>::N;
    const Slot<T> slot(rows);
    const size_t base = slot.row * width;
    Share<S, T, NV> r;
    r.place(slot.t, width, 0, (width + E - 1) / E);
    Vec16<S> wv[NV], rv[NV];
    r.params(w, wv);
    r.load(x + base);
    if constexpr (kResidual) {
#pragma unroll
        for (int j = 0; j < NV; ++j) rv[j] = load_any(residual + base + r.start[j]);
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < E; ++e)
                r.v[j].v[e] = Elem<S>::store(r.at(j, e) + Elem<S>::load(rv[j].v[e]));
    }
    float squares = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int e = 0; e < E; ++e) squares += r.counts(j, e) ? r.at(j, e) * r.at(j, e) : 0.0f;
    // the fold also orders every lane's loads before any store of the row, so
    // an output may be one of the inputs
    squares = row_total<T>(squares, lds);
    const float scale = 1.0f / sqrtf(squares / (float)width + eps);
    if constexpr (kResidual)
        r.store(sum_out + base, slot.live, [&](int j, int e) { return r.at(j, e); });
    r.store(y + base, slot.live,
            [&](int j, int e) { return r.at(j, e) * scale * Elem<S>::load(wv[j].v[e]); });
}

// Which of scale and bias there are (kEither: at run time; for one of them alone
// in rows of up to 4096 vectors, where it measured up to 10% faster at 512 rows
// than its own form, which keeps the longest rows within the registers).
enum Affine { kNeither = 0, kScaleOnly = 1, kBiasOnly = 2, kBoth = 3, kEither = 4 };

template <typename S, int T, int NV, int kAffine>
__global__ __launch_bounds__(block_threads<T>()) void layer_kernel(const S *x, const S *scale,
                                                                   const S *bias, S *y, size_t rows,
                                                                   uint32_t width, float eps) {
    __shared__ float lds[lds_floats<T>()];
    constexpr int E = Vec16<S>::N;
    const Slot<T> slot(rows);
    const size_t base = slot.row * width;
    Share<S, T, NV> r;
    r.place(slot.t, width, 0, (width + E - 1) / E);
    // the parameters' loads come first; the bias of the longest rows comes after
    // the sums (beside the row and the scale it does not fit the registers)
    constexpr bool kLate = T * NV > 4096;
    const bool has_scale = kAffine == kEither ? scale != nullptr : (kAffine & kScaleOnly) != 0;
    const bool has_bias = kAffine == kEither ? bias != nullptr : (kAffine & kBiasOnly) != 0;
    Vec16<S> sv[NV], bv[NV];
    if (has_scale) r.params(scale, sv);
    if (has_bias && !kLate) r.params(bias, bv);
    r.load(x + base);
    float total = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int e = 0; e < E; ++e) total += r.counts(j, e) ? r.at(j, e) : 0.0f;
    const float mean = row_total<T>(total, lds) / (float)width;
    float variance = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const float d = r.at(j, e) - mean;
            variance += r.counts(j, e) ? d * d : 0.0f;
        }
    variance = row_total<T>(variance, lds);
    const float inverse_std = 1.0f / sqrtf(variance / (float)width + eps);
    if (has_bias && kLate) r.params(bias, bv);
    r.store(y + base, slot.live, [&](int j, int e) {
        float v = (r.at(j, e) - mean) * inverse_std;
        if (has_scale) v *= Elem<S>::load(sv[j].v[e]);
        if (has_bias) v += Elem<S>::load(bv[j].v[e]);
        return v;
    });
}

// The rules of softmax_kernel (k_rowreduce.hip): a row whose maximum is -inf
// is zeros; +inf keys share the row; causal keys past the limit are -inf.
template <typename S, int T, int NV>
__global__ __launch_bounds__(block_threads<T>()) void softmax_kernel(const S *x, S *y, size_t rows,
                                                                     uint32_t width, size_t q_len,
                                                                     size_t offset) {
    __shared__ float lds[lds_floats<T>()];
    constexpr int E = Vec16<S>::N;
    const float inf = __builtin_inff();
    const Slot<T> slot(rows);
    const size_t base = slot.row * width;
    const uint32_t limit = causal_limit(slot.row, width, q_len, offset);
    Share<S, T, NV> r;
    r.place(slot.t, width, 0, (width + E - 1) / E);
    r.load(x + base);
    float p[NV][E];
    float m = -inf;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int e = 0; e < E; ++e) {
            p[j][e] = r.start[j] + e <= limit ? r.at(j, e) : -inf;
            m = fmaxf(m, p[j][e]);   // (an element counted twice does not move the maximum)
        }
    m = row_largest<T>(m, lds);
    float inverse = 0.0f, total = 1.0f;
    if (m == -inf) {
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < E; ++e) p[j][e] = 0.0f;
    } else if (m == inf) {
        float count = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < E; ++e) {
                p[j][e] = p[j][e] == inf ? 1.0f : 0.0f;
                count += r.counts(j, e) ? p[j][e] : 0.0f;
            }
        total = row_total<T>(count, lds);
    } else {
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < E; ++e) {
                p[j][e] = num_exp<S>(p[j][e] - m);
                sum += r.counts(j, e) ? p[j][e] : 0.0f;
            }
        total = row_total<T>(sum, lds);
    }
    inverse = 1.0f / total;
    r.store(y + base, slot.live, [&](int j, int e) {
        if constexpr (sizeof(S) == 2) return p[j][e] * inverse;
        else return p[j][e] / total;
    });
}

template <typename S, int T, int NV, bool kMax>
__global__ __launch_bounds__(block_threads<T>()) void reduce_kernel(const S *x, float *y, size_t rows,
                                                                    uint32_t width) {
    __shared__ float lds[lds_floats<T>()];
    constexpr int E = Vec16<S>::N;
    const Slot<T> slot(rows);
    Share<S, T, NV> r;
    r.place(slot.t, width, 0, (width + E - 1) / E);
    r.load(x + slot.row * width);
    float acc = kMax ? -__builtin_inff() : 0.0f, nans = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const float v = r.at(j, e);
            if constexpr (kMax) {
                acc = fmaxf(acc, v);
                nans = v != v ? 1.0f : nans;
            } else {
                acc += r.counts(j, e) ? v : 0.0f;
            }
        }
    float result = row_fold<T, kMax>(acc, lds);
    if constexpr (kMax) result = row_largest<T>(nans, lds) != 0.0f ? __builtin_nanf("") : result;
    if (slot.t == 0 && slot.live) y[slot.row] = result;
}

// ---- rows cut into parts over several blocks -----------------------------------------

// Vectors per part: kPartVectors at most, one less in the host's cut so that
// a last part of a single partial vector (whose overlap would lie in another
// block's part) can join the part before it.
constexpr int kPartThreads = 256, kPartNV = 8;
constexpr uint32_t kPartVectors = kPartThreads * kPartNV;

struct Cut {
    uint32_t parts, per;   // per: vectors of every part but the last
};

// This block's row and part, and its share of it.
template <typename S> struct PartShare {
    Share<S, kPartThreads, kPartNV> r;
    size_t row, base;
    uint32_t part, first, end;
    __device__ PartShare(uint32_t width, const Cut &c) {
        constexpr uint32_t E = Vec16<S>::N;
        row = blockIdx.x / c.parts;
        part = blockIdx.x % c.parts;
        base = row * width;
        const uint32_t vectors = (width + E - 1) / E;
        first = part * c.per;
        end = part + 1 == c.parts ? vectors : first + c.per;
        r.place(threadIdx.x, width, first, end);
    }
    __device__ inline uint32_t elements(uint32_t width) const {
        constexpr uint32_t E = Vec16<S>::N;
        return min(end * E, width) - first * E;
    }
};

enum class Op { kRms, kLayer, kSoftmax, kSum, kMax };

// A part's partial result: rms {sum of squares}, layer {sum, squares about the
// part's mean}, softmax {max, sum of exp(x - max), +inf keys}, sum {sum}, max
// {max, whether a NaN}.
template <typename S, Op kOp, bool kResidual>
__global__ __launch_bounds__(kPartThreads) void part_kernel(const S *x, const S *residual,
                                                            S *sum_out, f32x4 *partials,
                                                            uint32_t width, Cut cut, size_t q_len,
                                                            size_t offset) {
    __shared__ float lds[lds_floats<kPartThreads>()];
    constexpr int T = kPartThreads, NV = kPartNV, E = Vec16<S>::N;
    const float inf = __builtin_inff();
    PartShare<S> ps(width, cut);
    auto &r = ps.r;
    r.load(x + ps.base);
    if constexpr (kResidual) {
        Vec16<S> rv[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j) rv[j] = load_any(residual + ps.base + r.start[j]);
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < E; ++e)
                r.v[j].v[e] = Elem<S>::store(r.at(j, e) + Elem<S>::load(rv[j].v[e]));
        __syncthreads();   // sum_out may be x or the residual: every load before any store
        r.store(sum_out + ps.base, true, [&](int j, int e) { return r.at(j, e); });
    }
    f32x4 out = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (kOp == Op::kRms || kOp == Op::kSum || kOp == Op::kLayer) {
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const float v = r.at(j, e);
                acc += r.counts(j, e) ? (kOp == Op::kRms ? v * v : v) : 0.0f;
            }
        out.x = row_total<T>(acc, lds);
        if constexpr (kOp == Op::kLayer) {
            const float mean = out.x / (float)ps.elements(width);
            float about = 0.0f;
#pragma unroll
            for (int j = 0; j < NV; ++j)
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const float d = r.at(j, e) - mean;
                    about += r.counts(j, e) ? d * d : 0.0f;
                }
            out.y = row_total<T>(about, lds);
        }
    } else if constexpr (kOp == Op::kMax) {
        float acc = -inf, nans = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const float v = r.counts(j, e) ? r.at(j, e) : -inf;
                acc = fmaxf(acc, v);
                nans = v != v ? 1.0f : nans;
            }
        out.x = row_largest<T>(acc, lds);
        out.y = row_largest<T>(nans, lds);
    } else {
        const uint32_t limit = causal_limit(ps.row, width, q_len, offset);
        float m = -inf, count = 0.0f, nans = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const float s = r.counts(j, e) && r.start[j] + e <= limit ? r.at(j, e) : -inf;
                m = fmaxf(m, s);
                count += s == inf ? 1.0f : 0.0f;
                nans = s != s ? 1.0f : nans;
            }
        m = row_largest<T>(m, lds);
        float sum = 0.0f;
        // (a part with nothing but -inf and NaN keys: its sum is 0, or NaN if
        // it holds one; a part with a +inf key needs no sum)
        if (m == -inf) {
            sum = nans != 0.0f ? __builtin_nanf("") : 0.0f;
        } else if (m != inf) {
#pragma unroll
            for (int j = 0; j < NV; ++j)
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const bool use = r.counts(j, e) && r.start[j] + e <= limit;
                    sum += use ? num_exp<S>(r.at(j, e) - m) : 0.0f;
                }
        }
        out.x = m;
        out.y = row_total<T>(sum, lds);
        out.z = row_total<T>(count, lds);
    }
    if (threadIdx.x == 0) partials[blockIdx.x] = out;
}

// Folds a row's partials (every thread walks the row's parts at a stride of
// the block) and writes this block's part of the output; sum and max: one
// block per row, y the f32 results.
template <typename S, Op kOp>
__global__ __launch_bounds__(kPartThreads) void fold_kernel(const S *x, const S *scale,
                                                            const S *bias, S *y, float *reduced,
                                                            const f32x4 *partials, uint32_t width,
                                                            Cut cut, float eps, size_t q_len,
                                                            size_t offset) {
    __shared__ float lds[lds_floats<kPartThreads>()];
    constexpr int T = kPartThreads, NV = kPartNV, E = Vec16<S>::N;
    const float inf = __builtin_inff();
    constexpr bool kReduced = kOp == Op::kSum || kOp == Op::kMax;
    if constexpr (kReduced) {
        const f32x4 *mine = partials + (size_t)blockIdx.x * cut.parts;
        float acc = kOp == Op::kMax ? -inf : 0.0f, nans = 0.0f;
        for (uint32_t i = threadIdx.x; i < cut.parts; i += T) {
            const f32x4 v = mine[i];
            if constexpr (kOp == Op::kMax) {
                acc = fmaxf(acc, v.x);
                nans = v.y != 0.0f ? 1.0f : nans;
            } else {
                acc += v.x;
            }
        }
        float result = row_fold<T, kOp == Op::kMax>(acc, lds);
        if constexpr (kOp == Op::kMax)
            result = row_largest<T>(nans, lds) != 0.0f ? __builtin_nanf("") : result;
        if (threadIdx.x == 0) reduced[blockIdx.x] = result;
        return;
    } else {
        PartShare<S> ps(width, cut);
        auto &r = ps.r;
        const f32x4 *mine = partials + ps.row * cut.parts;
        r.load(x + ps.base);
        auto write = [&](auto &&value) {
            __syncthreads();   // y may be x: every load of the part before any store
            r.store(y + ps.base, true, value);
        };
        if constexpr (kOp == Op::kRms) {
            Vec16<S> wv[NV];
            r.params(scale, wv);
            float acc = 0.0f;
            for (uint32_t i = threadIdx.x; i < cut.parts; i += T) acc += mine[i].x;
            const float f = 1.0f / sqrtf(row_total<T>(acc, lds) / (float)width + eps);
            write([&](int j, int e) { return r.at(j, e) * f * Elem<S>::load(wv[j].v[e]); });
        } else if constexpr (kOp == Op::kLayer) {
            float acc = 0.0f;
            for (uint32_t i = threadIdx.x; i < cut.parts; i += T) acc += mine[i].x;
            const float mean = row_total<T>(acc, lds) / (float)width;
            // squares about the row's mean: about the part's, plus n (part
            // mean - mean)^2
            const float n_part = (float)(cut.per * E);
            float about = 0.0f;
            for (uint32_t i = threadIdx.x; i < cut.parts; i += T) {
                const float n = i + 1 == cut.parts ? (float)(width - i * cut.per * E) : n_part;
                const float d = mine[i].x / n - mean;
                about += mine[i].y + n * d * d;
            }
            const float inverse_std = 1.0f / sqrtf(row_total<T>(about, lds) / (float)width + eps);
            Vec16<S> sv[NV], bv[NV];
            if (scale) r.params(scale, sv);
            if (bias) r.params(bias, bv);
            write([&](int j, int e) {
                float v = (r.at(j, e) - mean) * inverse_std;
                if (scale) v *= Elem<S>::load(sv[j].v[e]);
                if (bias) v += Elem<S>::load(bv[j].v[e]);
                return v;
            });
        } else {
            float m = -inf;
            for (uint32_t i = threadIdx.x; i < cut.parts; i += T) m = fmaxf(m, mine[i].x);
            m = row_largest<T>(m, lds);
            const uint32_t limit = causal_limit(ps.row, width, q_len, offset);
            if (m == -inf) {
                write([&](int, int) { return 0.0f; });
                return;
            }
            float acc = 0.0f;
            for (uint32_t i = threadIdx.x; i < cut.parts; i += T) {
                const f32x4 v = mine[i];
                acc += m == inf ? v.z : v.x == -inf ? v.y : v.y * num_exp<S>(v.x - m);
            }
            const float total = row_total<T>(acc, lds);
            const float inverse = 1.0f / total;
            write([&](int j, int e) {
                const float s = r.start[j] + e <= limit ? r.at(j, e) : -inf;
                const float p = m == inf ? (s == inf ? 1.0f : 0.0f) : num_exp<S>(s - m);
                if constexpr (sizeof(S) == 2) return p * inverse;
                else return p / total;
            });
        }
    }
}

// ---- launch shapes ---------------------------------------------------------------------

// Lanes and vectors per lane for a row of `vectors` vectors, or 0 lanes where
// the row is cut into parts. A second launch costs about 2.5 us (one row of
// 32000 f32: 7.5 us cut, 5 in one block), so rows of up to 4096 vectors stay
// whole; f32 rows of up to 8192 too where there are enough of them to fill
// the chip (f16 rows of that length do not fit the registers with their
// parameters).
struct Shape {
    int t, nv;
};

inline Shape pick(size_t vectors, size_t rows, size_t elem) {
    if (vectors <= 8) return {8, 1};
    if (vectors <= 16) return {16, 1};
    if (vectors <= 32) return {32, 1};
    if (vectors <= 64) return {64, 1};
    if (vectors <= 128) return {64, 2};
    if (vectors <= 256) return {256, 1};
    if (vectors <= 512) return {256, 2};
    if (vectors <= 1024) return {256, 4};
    if (vectors <= 2048) return {256, 8};
    if (vectors <= 4096) return {1024, 4};
    if (vectors <= 8192 && elem == 4 && rows >= 128) return {1024, 8};
    return {0, 0};
}

inline size_t blocks_for(const Shape &sh, size_t rows) {
    const size_t per = sh.t > kWave ? 1 : kBlock / sh.t;
    return (rows + per - 1) / per;
}

// The cut of a row into parts of at most kPartVectors vectors, the last of at
// least two where there are several.
inline Cut cut_row(size_t vectors) {
    Cut c;
    c.parts = (uint32_t)((vectors + kPartVectors - 2) / (kPartVectors - 1));
    c.per = (uint32_t)((vectors + c.parts - 1) / c.parts);
    c.parts = (uint32_t)((vectors + c.per - 1) / c.per);
    if (c.parts > 1 && vectors - (size_t)(c.parts - 1) * c.per < 2) --c.parts;
    return c;
}

struct Plan {
    Shape shape;
    Cut cut;
    size_t blocks;
    bool ok;
};

template <typename S> Plan plan_row(size_t rows, size_t width) {
    constexpr size_t E = Vec16<S>::N;
    Plan p{{0, 0}, {0, 0}, 0, false};
    if (width < E || width > 0xfffffff0u) return p;
    const size_t vectors = (width + E - 1) / E;
    p.shape = pick(vectors, rows, sizeof(S));
    if (p.shape.t != 0) {
        p.blocks = blocks_for(p.shape, rows);
    } else {
        if (sdk_recording() != Recording::kNo) return p;   // one kernel and no memory in a graph
        p.cut = cut_row(vectors);
        p.blocks = rows * p.cut.parts;
    }
    const size_t threads = p.shape.t > kBlock ? p.shape.t : kBlock;
    p.ok = p.blocks <= 0xffffffffu / threads;
    return p;
}

#define ICSDK_ANY_DISPATCH(shape, CASE)              \
    do {                                             \
        switch ((shape).t * 10 + (shape).nv) {       \
            case 81: CASE(8, 1); break;              \
            case 161: CASE(16, 1); break;            \
            case 321: CASE(32, 1); break;            \
            case 641: CASE(64, 1); break;            \
            case 642: CASE(64, 2); break;            \
            case 2561: CASE(256, 1); break;          \
            case 2562: CASE(256, 2); break;          \
            case 2564: CASE(256, 4); break;          \
            case 2568: CASE(256, 8); break;          \
            case 10244: CASE(1024, 4); break;        \
            case 10248:                              \
                if constexpr (sizeof(S) == 4) {      \
                    CASE(1024, 8);                   \
                    break;                           \
                }                                    \
                return hipErrorInvalidValue;         \
            default: return hipErrorInvalidValue;    \
        }                                            \
        return hipGetLastError();                    \
    } while (0)

}  // namespace

template <typename S>
hipError_t rms_norm(const S *x, const S *residual, S *sum_out, const S *w, S *y, size_t rows,
                    size_t width, float eps, hipStream_t s) {
    const Plan p = plan_row<S>(rows, width);
    if (!p.ok) return hipErrorNotSupported;
    const dim3 grid((unsigned)p.blocks);
#define ICSDK_CASE(T, NV)                                                                        \
    do {                                                                                         \
        if (residual)                                                                            \
            hipLaunchKernelGGL((rms_kernel<S, T, NV, true>), grid, dim3(block_threads<T>()), 0,  \
                               s, x, residual, sum_out, w, y, rows, (uint32_t)width, eps);       \
        else                                                                                     \
            hipLaunchKernelGGL((rms_kernel<S, T, NV, false>), grid, dim3(block_threads<T>()), 0, \
                               s, x, residual, sum_out, w, y, rows, (uint32_t)width, eps);       \
    } while (0)
    if (p.shape.t != 0) ICSDK_ANY_DISPATCH(p.shape, ICSDK_CASE);
#undef ICSDK_CASE
    ScratchBlock scratch(p.blocks * sizeof(f32x4));
    if (scratch.get() == nullptr) return hipErrorNotSupported;
    f32x4 *partials = static_cast<f32x4 *>(scratch.get());
    if (residual)
        hipLaunchKernelGGL((part_kernel<S, Op::kRms, true>), grid, dim3(kPartThreads), 0, s, x,
                           residual, sum_out, partials, (uint32_t)width, p.cut, (size_t)0, (size_t)0);
    else
        hipLaunchKernelGGL((part_kernel<S, Op::kRms, false>), grid, dim3(kPartThreads), 0, s, x,
                           residual, sum_out, partials, (uint32_t)width, p.cut, (size_t)0, (size_t)0);
    hipLaunchKernelGGL((fold_kernel<S, Op::kRms>), grid, dim3(kPartThreads), 0, s,
                       residual ? sum_out : x, w, (const S *)nullptr, y, (float *)nullptr, partials,
                       (uint32_t)width, p.cut, eps, (size_t)0, (size_t)0);
    return hipGetLastError();
}

template <typename S>
hipError_t layer_norm(const S *x, const S *scale, const S *bias, S *y, size_t rows, size_t width,
                      float eps, hipStream_t s) {
    const Plan p = plan_row<S>(rows, width);
    if (!p.ok) return hipErrorNotSupported;
    const dim3 grid((unsigned)p.blocks);
#define ICSDK_LAYER(T, NV, AFFINE)                                                           \
    hipLaunchKernelGGL((layer_kernel<S, T, NV, AFFINE>), grid, dim3(block_threads<T>()), 0, s, x, \
                       scale, bias, y, rows, (uint32_t)width, eps)
#define ICSDK_CASE(T, NV)                                                             \
    do {                                                                              \
        if (scale && bias) ICSDK_LAYER(T, NV, kBoth);                                 \
        else if (scale) ICSDK_LAYER(T, NV, (T * NV > 4096 ? kScaleOnly : kEither));   \
        else if (bias) ICSDK_LAYER(T, NV, (T * NV > 4096 ? kBiasOnly : kEither));     \
        else ICSDK_LAYER(T, NV, kNeither);                                            \
    } while (0)
    if (p.shape.t != 0) ICSDK_ANY_DISPATCH(p.shape, ICSDK_CASE);
#undef ICSDK_CASE
#undef ICSDK_LAYER
    ScratchBlock scratch(p.blocks * sizeof(f32x4));
    if (scratch.get() == nullptr) return hipErrorNotSupported;
    f32x4 *partials = static_cast<f32x4 *>(scratch.get());
    hipLaunchKernelGGL((part_kernel<S, Op::kLayer, false>), grid, dim3(kPartThreads), 0, s, x,
                       (const S *)nullptr, (S *)nullptr, partials, (uint32_t)width, p.cut, (size_t)0,
                       (size_t)0);
    hipLaunchKernelGGL((fold_kernel<S, Op::kLayer>), grid, dim3(kPartThreads), 0, s, x, scale, bias, y,
                       (float *)nullptr, partials, (uint32_t)width, p.cut, eps, (size_t)0, (size_t)0);
    return hipGetLastError();
}

template <typename S>
hipError_t softmax(const S *x, S *y, size_t rows, size_t width, size_t q_len,
                   size_t causal_offset, hipStream_t s) {
    const Plan p = plan_row<S>(rows, width);
    if (!p.ok) return hipErrorNotSupported;
    const dim3 grid((unsigned)p.blocks);
#define ICSDK_CASE(T, NV)                                                                       \
    hipLaunchKernelGGL((softmax_kernel<S, T, NV>), grid, dim3(block_threads<T>()), 0, s, x, y, \
                       rows, (uint32_t)width, q_len, causal_offset)
    if (p.shape.t != 0) ICSDK_ANY_DISPATCH(p.shape, ICSDK_CASE);
#undef ICSDK_CASE
    ScratchBlock scratch(p.blocks * sizeof(f32x4));
    if (scratch.get() == nullptr) return hipErrorNotSupported;
    f32x4 *partials = static_cast<f32x4 *>(scratch.get());
    hipLaunchKernelGGL((part_kernel<S, Op::kSoftmax, false>), grid, dim3(kPartThreads), 0, s, x,
                       (const S *)nullptr, (S *)nullptr, partials, (uint32_t)width, p.cut, q_len,
                       causal_offset);
    hipLaunchKernelGGL((fold_kernel<S, Op::kSoftmax>), grid, dim3(kPartThreads), 0, s, x,
                       (const S *)nullptr, (const S *)nullptr, y, (float *)nullptr, partials,
                       (uint32_t)width, p.cut, 0.0f, q_len, causal_offset);
    return hipGetLastError();
}

template <typename S, bool kMax>
hipError_t reduce(const S *x, float *y, size_t rows, size_t width, hipStream_t s) {
    const Plan p = plan_row<S>(rows, width);
    if (!p.ok) return hipErrorNotSupported;
    const dim3 grid((unsigned)p.blocks);
#define ICSDK_CASE(T, NV)                                                                       \
    hipLaunchKernelGGL((reduce_kernel<S, T, NV, kMax>), grid, dim3(block_threads<T>()), 0, s, x, \
                       y, rows, (uint32_t)width)
    if (p.shape.t != 0) ICSDK_ANY_DISPATCH(p.shape, ICSDK_CASE);
#undef ICSDK_CASE
    constexpr Op kOp = kMax ? Op::kMax : Op::kSum;
    ScratchBlock scratch(p.blocks * sizeof(f32x4));
    if (scratch.get() == nullptr) return hipErrorNotSupported;
    f32x4 *partials = static_cast<f32x4 *>(scratch.get());
    hipLaunchKernelGGL((part_kernel<S, kOp, false>), grid, dim3(kPartThreads), 0, s, x,
                       (const S *)nullptr, (S *)nullptr, partials, (uint32_t)width, p.cut, (size_t)0,
                       (size_t)0);
    hipLaunchKernelGGL((fold_kernel<S, kOp>), dim3((unsigned)rows), dim3(kPartThreads), 0, s, x,
                       (const S *)nullptr, (const S *)nullptr, (S *)nullptr, y, partials,
                       (uint32_t)width, p.cut, 0.0f, (size_t)0, (size_t)0);
    return hipGetLastError();
}

#undef ICSDK_ANY_DISPATCH

#define ICSDK_INSTANTIATE(S)                                                                       \
    template hipError_t rms_norm<S>(const S *, const S *, S *, const S *, S *, size_t, size_t,     \
                                    float, hipStream_t);                                           \
    template hipError_t layer_norm<S>(const S *, const S *, const S *, S *, size_t, size_t, float, \
                                      hipStream_t);                                                \
    template hipError_t softmax<S>(const S *, S *, size_t, size_t, size_t, size_t, hipStream_t);   \
    template hipError_t reduce<S, false>(const S *, float *, size_t, size_t, hipStream_t);         \
    template hipError_t reduce<S, true>(const S *, float *, size_t, size_t, hipStream_t);
ICSDK_INSTANTIATE(float)
ICSDK_INSTANTIATE(_Float16)
#undef ICSDK_INSTANTIATE

}  // namespace row_any
}  // namespace icsdk
