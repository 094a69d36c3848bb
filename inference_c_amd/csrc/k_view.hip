// Strided view with broadcast operands for gfx950:
//     y[i] = (x[view(i)] + addend[bcast(i)]) * mult[bcast(i)]
// with y contiguous in the view's shape.
//
// The host first coalesces the view: dimensions of extent 1 are dropped and a
// dimension is merged into its inner neighbour when x, the addend and the
// multiplier all step through both as through one (a contiguous tensor
// becomes rank 1, a (0,2,1,3) permutation stays rank 4). Then one of three
// paths runs, chosen from the coalesced strides:
//   gather  - the innermost dimension is contiguous in x and every offset is
//             a multiple of the 16-byte vector. One output vector per lane on
//             a one-shot grid: the block's outer coordinates are decomposed
//             once per block, the lane adds its (row, vector) offsets, loads
//             one 16-byte run of x, applies the broadcast operands (a vector
//             where the operand varies along the innermost dimension, a
//             scalar where it is broadcast along it) and stores 16 bytes
//             through L2. Each run is a whole contiguous vector, so no loaded
//             byte is wasted and no staging is needed; measured on MI355X
//             this beats staging the same permutation through LDS tiles at
//             every run length from 16 to 256 bytes;
//   tile    - x's contiguous dimension is another view dimension p (a
//             transpose of p with the innermost dimension): tiles are read
//             along p, staged through LDS (swizzled or padded against bank
//             conflicts) and written along the innermost dimension, so both
//             HBM streams stay coalesced: 64x64 tiles in 16-byte vectors of
//             any alignment where both dimensions have 64 elements (whole
//             aligned vectors also with fewer), else tiles of about 4096 or
//             1024 elements shaped to the smaller one;
//   scalar  - anything else, and transposes that would leave a tile mostly
//             empty: one element per lane.
#include "kern_common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>

namespace icsdk {
namespace {

constexpr int kMaxRank = 8;

// The view after coalescing (element strides; 0 where an operand broadcasts).
struct Coalesced {
    int rank;
    uint64_t shape[kMaxRank];
    int64_t x_stride[kMaxRank];
    uint64_t a_stride[kMaxRank];
    uint64_t m_stride[kMaxRank];
};

// Contiguous strides of a broadcast operand, zeroed where its dim is 1.
inline void broadcast_strides(const uint64_t *shape, int rank, uint64_t *out) {
    uint64_t s = 1;
    for (int d = rank - 1; d >= 0; --d) {
        out[d] = shape[d] == 1 ? 0 : s;
        s *= shape[d];
    }
}

Coalesced coalesce(const k::ViewArgs &v, const uint64_t *a_stride, const uint64_t *m_stride) {
    Coalesced c{};
    // walk from the innermost dimension outwards, building c back to front
    int r = 0;
    uint64_t shape[kMaxRank];
    int64_t xs[kMaxRank];
    uint64_t as[kMaxRank], ms[kMaxRank];
    for (int d = v.rank - 1; d >= 0; --d) {
        if (v.shape[d] == 1) continue;
        if (r > 0) {
            const int in = r - 1;
            const bool merge = v.strides[d] == xs[in] * (int64_t)shape[in] &&
                               a_stride[d] == as[in] * shape[in] &&
                               m_stride[d] == ms[in] * shape[in];
            if (merge) {
                shape[in] *= v.shape[d];
                continue;
            }
        }
        shape[r] = v.shape[d];
        xs[r] = v.strides[d];
        as[r] = a_stride[d];
        ms[r] = m_stride[d];
        ++r;
    }
    if (r == 0) {  // every extent is 1
        shape[0] = 1;
        xs[0] = 1;
        as[0] = ms[0] = 0;
        r = 1;
    }
    c.rank = r;
    for (int i = 0; i < r; ++i) {
        c.shape[i] = shape[r - 1 - i];
        c.x_stride[i] = xs[r - 1 - i];
        c.a_stride[i] = as[r - 1 - i];
        c.m_stride[i] = ms[r - 1 - i];
    }
    return c;
}

// ---- gather path -------------------------------------------------------------

// The coalesced view is split into outer dims 0..R-3 and an inner plane of
// dims R-2 (rows) and R-1 (runs, counted in 16-byte vectors). A block covers
// kBlock consecutive vectors of one inner plane: its outer coordinates and
// their offsets are decomposed once per block from blockIdx (block-uniform,
// so the compiler keeps them in scalar registers and off the vector ALU),
// and each lane only splits its plane index into (row, vector) and adds two
// products per operand, in 32 bits. The quarter-rate 32-bit multiplies of a
// full per-lane decomposition otherwise sit between every lane and its load.
struct GatherPlan {
    int outer_rank;                // dims 0..outer_rank-1 (R - 2, or 0)
    FastDiv outer[kMaxRank];       // their extents
    uint64_t ox[kMaxRank], oa[kMaxRank], om[kMaxRank];  // their element strides
    FastDiv plane_blocks;          // blocks per inner plane
    FastDiv vecs;                  // vectors per row (innermost extent / E)
    int vecs_log2;                 // log2(vecs) when vecs is a power of two, else -1
    uint32_t plane;                // vectors per inner plane (rows * vecs)
    uint32_t row_x, row_a, row_m;  // element strides of the row dim
    uint64_t x_offset;
};

// How a broadcast operand enters: absent, one 16-byte vector per output
// vector (it varies along the innermost dimension) or one element per output
// vector (broadcast along it). A compile-time choice, so that every load of
// the kernel is unconditional: a load behind a run-time branch is followed by
// a wait for all outstanding loads, which would serialise the three streams.
enum OperandKind { kNone = 0, kVector = 1, kScalar = 2 };

template <typename S, int kA, int kM>
__global__ __launch_bounds__(kBlock) void view_gather_kernel(const S *__restrict__ x,
                                                             const S *__restrict__ addend,
                                                             const S *__restrict__ mult,
                                                             S *__restrict__ y,
                                                             GatherPlan plan) {
    constexpr int E = Vec16<S>::N;
    // block-uniform part
    const uint32_t b = blockIdx.x;
    uint32_t outer = fast_div(b, plan.plane_blocks);
    const uint32_t in_block = b - outer * plan.plane_blocks.divisor;
    const uint64_t out_vec0 = (uint64_t)outer * plan.plane + (uint64_t)in_block * kBlock;
    uint64_t xb = plan.x_offset, ab = 0, mb = 0;
    for (int d = plan.outer_rank - 1; d >= 0; --d) {
        uint32_t idx = outer;
        if (d > 0) {
            const uint32_t q = fast_div(outer, plan.outer[d]);
            idx = outer - q * plan.outer[d].divisor;
            outer = q;
        }
        xb += idx * plan.ox[d];
        ab += idx * plan.oa[d];
        mb += idx * plan.om[d];
    }
    // lane part
    const uint32_t t = in_block * kBlock + threadIdx.x;  // vector index inside the plane
    if (t >= plan.plane) return;
    const uint32_t row = plan.vecs_log2 >= 0 ? t >> plan.vecs_log2 : fast_div(t, plan.vecs);
    const uint32_t vec = t - row * plan.vecs.divisor;
    const Vec16<S> xv = load16_stream(x + xb + (row * plan.row_x + vec * E));
    Vec16<S> av, mv;
    float a_scalar = 0.0f, m_scalar = 1.0f;
    if constexpr (kA == kVector) av = load16(addend + ab + (row * plan.row_a + vec * E));
    if constexpr (kA == kScalar) a_scalar = Elem<S>::load(addend[ab + row * plan.row_a]);
    if constexpr (kM == kVector) mv = load16(mult + mb + (row * plan.row_m + vec * E));
    if constexpr (kM == kScalar) m_scalar = Elem<S>::load(mult[mb + row * plan.row_m]);
    Vec16<S> out;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        float r = Elem<S>::load(xv.v[e]);
        if constexpr (kA != kNone) r = r + (kA == kVector ? Elem<S>::load(av.v[e]) : a_scalar);
        if constexpr (kM != kNone) r = r * (kM == kVector ? Elem<S>::load(mv.v[e]) : m_scalar);
        out.v[e] = Elem<S>::store(r);
    }
    const OutWindow window(y + out_vec0 * E, kBlock * 16u);
    window.store16(threadIdx.x * 16u, out);
}

// Short gather: the common views -- at most two outer dims, whole blocks of
// kBlock vectors per inner plane, a power-of-two number of vectors per row,
// and every element offset below 2^32. The outer coordinates are blockIdx.z
// and blockIdx.y (a 3-D grid), strides are 32-bit, the row split is a shift
// and there is no bounds test: a wave reaches its loads after a few
// independent scalar loads instead of the general plan's chain of dependent
// ones (config-4 shape, measured in isolation: 23.6 -> 22.7 us).
struct ShortPlan {
    uint32_t ox[2], oa[2], om[2];  // element strides of the outer dims (grid z, y)
    uint32_t x_offset;
    uint32_t vecs_log2;            // log2(vectors per row)
    uint32_t row_x, row_a, row_m;  // element strides of the row dim
};

template <typename S, int kA, int kM>
__global__ __launch_bounds__(kBlock) void view_gather_short_kernel(const S *__restrict__ x,
                                                                   const S *__restrict__ addend,
                                                                   const S *__restrict__ mult,
                                                                   S *__restrict__ y,
                                                                   ShortPlan plan) {
    constexpr int E = Vec16<S>::N;
    const uint32_t xb = plan.x_offset + blockIdx.z * plan.ox[0] + blockIdx.y * plan.ox[1];
    const uint32_t ab = blockIdx.z * plan.oa[0] + blockIdx.y * plan.oa[1];
    const uint32_t mb = blockIdx.z * plan.om[0] + blockIdx.y * plan.om[1];
    const uint32_t plane_vec0 = blockIdx.x * kBlock;
    const size_t out_vec0 = ((size_t)blockIdx.z * gridDim.y + blockIdx.y) * (gridDim.x * kBlock) +
                            plane_vec0;
    const uint32_t t = plane_vec0 + threadIdx.x;
    const uint32_t row = t >> plan.vecs_log2;
    const uint32_t vec = t - (row << plan.vecs_log2);
    const Vec16<S> xv = load16_stream(x + (xb + row * plan.row_x + vec * E));
    Vec16<S> av, mv;
    float a_scalar = 0.0f, m_scalar = 1.0f;
    if constexpr (kA == kVector) av = load16(addend + (ab + row * plan.row_a + vec * E));
    if constexpr (kA == kScalar) a_scalar = Elem<S>::load(addend[ab + row * plan.row_a]);
    if constexpr (kM == kVector) mv = load16(mult + (mb + row * plan.row_m + vec * E));
    if constexpr (kM == kScalar) m_scalar = Elem<S>::load(mult[mb + row * plan.row_m]);
    Vec16<S> out;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        float r = Elem<S>::load(xv.v[e]);
        if constexpr (kA != kNone) r = r + (kA == kVector ? Elem<S>::load(av.v[e]) : a_scalar);
        if constexpr (kM != kNone) r = r * (kM == kVector ? Elem<S>::load(mv.v[e]) : m_scalar);
        out.v[e] = Elem<S>::store(r);
    }
    const OutWindow window(y + out_vec0 * E, kBlock * 16u);
    window.store16(threadIdx.x * 16u, out);
}

// The short plan of a view the gather path takes, or false when the view
// needs the general kernel.
template <typename S>
bool short_plan(const Coalesced &c, uint64_t x_offset, uint64_t n, ShortPlan *plan, dim3 *grid) {
    constexpr uint64_t E = Vec16<S>::N;
    const int last = c.rank - 1;
    const int outer_rank = c.rank >= 2 ? c.rank - 2 : 0;
    if (outer_rank > 2 || n > 0xffffffffull) return false;
    // offsets are unsigned 32-bit sums: a negative stride would make the
    // reach below wrap (and the base offset be truncated) undetected
    for (int d = 0; d < c.rank; ++d)
        if (c.x_stride[d] < 0) return false;
    const uint64_t vecs = c.shape[last] / E;
    const uint64_t rows = c.rank >= 2 ? c.shape[last - 1] : 1;
    const uint64_t plane = rows * vecs;
    if ((vecs & (vecs - 1)) != 0 || plane % kBlock != 0 || plane / kBlock > 0x7fffffffull)
        return false;
    uint64_t ext[2] = {1, 1}, ox[2] = {0, 0}, oa[2] = {0, 0}, om[2] = {0, 0};
    for (int d = 0; d < outer_rank; ++d) {
        const int slot = 2 - outer_rank + d;
        ext[slot] = c.shape[d];
        ox[slot] = (uint64_t)c.x_stride[d];
        oa[slot] = c.a_stride[d];
        om[slot] = c.m_stride[d];
    }
    if (ext[0] > 65535 || ext[1] > 65535) return false;
    const uint64_t row_x = c.rank >= 2 ? (uint64_t)c.x_stride[last - 1] : 0;
    const uint64_t row_a = c.rank >= 2 ? c.a_stride[last - 1] : 0;
    const uint64_t row_m = c.rank >= 2 ? c.m_stride[last - 1] : 0;
    // the largest element offset each operand is addressed at, in 32 bits
    auto reach = [&](uint64_t base, const uint64_t (&o)[2], uint64_t row, uint64_t inner) {
        return base + (ext[0] - 1) * o[0] + (ext[1] - 1) * o[1] + (rows - 1) * row + inner;
    };
    if (reach(x_offset, ox, row_x, vecs * E) > 0xffffffffull ||
        reach(0, oa, row_a, vecs * E) > 0xffffffffull || reach(0, om, row_m, vecs * E) > 0xffffffffull)
        return false;
    *plan = ShortPlan{{(uint32_t)ox[0], (uint32_t)ox[1]}, {(uint32_t)oa[0], (uint32_t)oa[1]},
                      {(uint32_t)om[0], (uint32_t)om[1]}, (uint32_t)x_offset,
                      (uint32_t)__builtin_ctzll(vecs), (uint32_t)row_x, (uint32_t)row_a,
                      (uint32_t)row_m};
    *grid = dim3((unsigned)(plane / kBlock), (unsigned)ext[1], (unsigned)ext[0]);
    return true;
}

// ---- scalar path -------------------------------------------------------------

// The product as the f32 value it is. (The compiler otherwise folds a f32
// multiply and its conversion to f16 into v_fma_mixlo_f16, which rounds once:
// another result at ties.)
template <typename S> __device__ inline float rounded_f32(float v) {
    if constexpr (sizeof(S) == 2) asm("" : "+v"(v));
    return v;
}

struct ScalarPlan {
    int rank;
    uint64_t shape[kMaxRank];
    int64_t x_stride[kMaxRank];
    uint64_t a_stride[kMaxRank];
    uint64_t m_stride[kMaxRank];
    uint64_t x_offset;
};

template <typename S>
__global__ __launch_bounds__(kBlock) void view_scalar_kernel(const S *__restrict__ x,
                                                             const S *__restrict__ addend,
                                                             const S *__restrict__ mult,
                                                             S *__restrict__ y, size_t n,
                                                             ScalarPlan plan) {
    const size_t stride = (size_t)gridDim.x * kBlock;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += stride) {
        size_t rest = i;
        int64_t xo = (int64_t)plan.x_offset;
        uint64_t ao = 0, mo = 0;
        for (int d = plan.rank - 1; d >= 0; --d) {
            const uint64_t idx = rest % plan.shape[d];
            rest /= plan.shape[d];
            xo += (int64_t)idx * plan.x_stride[d];
            ao += idx * plan.a_stride[d];
            mo += idx * plan.m_stride[d];
        }
        float r = Elem<S>::load(x[xo]);
        if (addend) r = r + Elem<S>::load(addend[ao]);
        if (mult) r = rounded_f32<S>(r * Elem<S>::load(mult[mo]));
        y[i] = Elem<S>::store(r);
    }
}

// ---- LDS-tiled transpose path ------------------------------------------------

// Output dims are viewed as [outer..., P, inner..., L] where dimension p has
// x stride 1 and L is the last view dimension. A block moves one tile of (p,
// last) for one combination of the remaining indices ("batch").
constexpr int kTile = 64;
constexpr uint32_t kTileElems = 4096;      // elements per block of the adaptive tiles, or
constexpr uint32_t kTileElemsSmall = 1024; // for small views

struct TilePlan {
    int rank;
    int p;                          // view dim with x stride 1
    uint64_t shape[kMaxRank];
    int64_t x_stride[kMaxRank];
    uint64_t a_stride[kMaxRank];
    uint64_t m_stride[kMaxRank];
    uint64_t y_stride[kMaxRank];    // contiguous output strides
    uint64_t x_offset;
    uint64_t batches;               // product of the dims other than p and last
    uint32_t tiles_p, tiles_l;
    FastDiv tile_p, tile_l;         // the adaptive tile's extents
};

// Where a batch starts in each operand.
struct BatchBase {
    int64_t x;
    uint64_t a, m, y;
    __device__ BatchBase(const TilePlan &plan, uint64_t batch)
        : x((int64_t)plan.x_offset), a(0), m(0), y(0) {
        if (batch == 0) return;   // block-uniform
        for (int d = plan.rank - 2; d >= 0; --d) {
            if (d == plan.p) continue;
            const uint64_t idx = batch % plan.shape[d];
            batch /= plan.shape[d];
            x += (int64_t)idx * plan.x_stride[d];
            a += idx * plan.a_stride[d];
            m += idx * plan.m_stride[d];
            y += idx * plan.y_stride[d];
        }
    }
};

// Tiles of tile_p x tile_l elements, about kTileElems in all: with a short p
// (the channels of an image stored channel-last) or a short last dimension
// the other one is long, so a block still moves 4096 elements and both its
// reads and its writes run along memory. One element per lane and access, 16
// of each lane in flight; reads past the tile are clamped onto its first
// element and not stored. LDS rows [l], pitch odd: conflict-free both ways.
// NHWC [8, 512, 512, 3] f32 to NCHW 117 -> 11.7 us, with both operands 122 ->
// 16.4 (64 x 64 tiles, 61 of 64 columns empty, before).
template <typename S, uint32_t kElems, bool kA, bool kM>
__global__ __launch_bounds__(kBlock) void view_tile_kernel(const S *__restrict__ x,
                                                           const S *__restrict__ addend,
                                                           const S *__restrict__ mult,
                                                           S *__restrict__ y, TilePlan plan) {
    __shared__ S tile[kElems / 2 * 3];   // tile_l * pitch (the host checks)
    constexpr int kPer = kElems / kBlock;
    const int last = plan.rank - 1;
    const uint64_t block = blockIdx.x;
    const uint32_t tl = (uint32_t)(block % plan.tiles_l);
    const uint32_t tp = (uint32_t)((block / plan.tiles_l) % plan.tiles_p);
    const BatchBase base(plan, block / ((uint64_t)plan.tiles_l * plan.tiles_p));
    const uint32_t ep = plan.tile_p.divisor, el = plan.tile_l.divisor, pitch = ep | 1u;
    const uint64_t p0 = (uint64_t)tp * ep, l0 = (uint64_t)tl * el;
    const uint32_t np = (uint32_t)min((uint64_t)ep, plan.shape[plan.p] - p0);
    const uint32_t nl = (uint32_t)min((uint64_t)el, plan.shape[last] - l0);
    // read: consecutive lanes walk p (contiguous in x), then l
    const int64_t xl = plan.x_stride[last];
    const S *xt = x + base.x + (int64_t)p0 + (int64_t)l0 * xl;
    S v[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const uint32_t t = threadIdx.x + k * kBlock, l = fast_div(t, plan.tile_p), p = t - l * ep;
        v[k] = xt[p < np && l < nl ? (int64_t)l * xl + p : 0];
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const uint32_t t = threadIdx.x + k * kBlock, l = fast_div(t, plan.tile_p), p = t - l * ep;
        if (l < el) tile[l * pitch + p] = v[k];
    }
    __syncthreads();
    // write: consecutive lanes walk the last dim (contiguous in y), then p
    const uint64_t ap = plan.a_stride[plan.p], al = plan.a_stride[last];
    const uint64_t mp = plan.m_stride[plan.p], ml = plan.m_stride[last], yp = plan.y_stride[plan.p];
    const S *at = kA ? addend + base.a + p0 * ap + l0 * al : nullptr;
    const S *mt = kM ? mult + base.m + p0 * mp + l0 * ml : nullptr;
    S *yt = y + base.y + p0 * yp + l0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        const uint32_t t = threadIdx.x + k * kBlock, p = fast_div(t, plan.tile_l), l = t - p * el;
        const bool in = p < np && l < nl;
        float r = Elem<S>::load(tile[in ? l * pitch + p : 0]);
        if constexpr (kA) r = r + Elem<S>::load(at[in ? p * ap + l * al : 0]);
        if constexpr (kM) r = rounded_f32<S>(r * Elem<S>::load(mt[in ? p * mp + l * ml : 0]));
        if (in) yt[p * yp + l] = Elem<S>::store(r);
    }
}

// 64 x 64 tiles in 16-byte vectors of E elements (8 for f16, 4 for f32), for
// views whose p and last dimensions have at least 64 elements: a tile's 64 x
// rows (64 elements along p, contiguous in x) are read as 64 / E vectors each
// into LDS rows [l], vector c of row l at slot c ^ (l / E); each output row (64
// elements along the last dim, contiguous in y) is gathered from one LDS
// column, E reads per vector, and written as 64 / E vectors. With the slot
// swizzle the 64 lanes of a gather read distinct banks (f16: 32, lanes 2m and
// 2m + 1 sharing a dword; f32: 64). A last tile that would reach past the end
// starts 64 elements before it instead and writes the overlap with the same
// values, so no access needs a bounds test; vectors are loaded and stored at
// any element alignment. A block takes kTiles tiles along the last dim: two for
// f16 where that still leaves 1024 blocks, else one (f16 with an addend, one /
// two / four tiles: [3000, 3000] 13.7 / 10.0 / 11.3 us, [8192, 8192] 48.9 /
// 47.0 / 47.9, [4096, 4096] 13.4 / 15.0 / 16.4). kGuarded: the form for whole
// aligned vectors without operands: bounds tests instead of the overlap (the
// launcher says where), f16 with four tiles, each load waited for before the
// next, which is the faster one there ([4096, 4000] 11.6 us against 12.7-12.8,
// [64, 512, 512] 12.4 against 13.2-15.6). Operands enter as a vector along the
// last dim or as one element per output row (OperandKind), loaded before the
// barrier. Against the one-element-per-lane tiles: f16 [4097, 4095] 30.0 ->
// 21.4 us, [4096, 4096] with both operands 41.0 -> 15.1, f32 39.6 -> 26.0.
//
// Everything a wave needs before its first load arrives as a plain scalar
// argument (preloaded in SGPRs; the tile grid split by multiply-high
// divisions); the plan is read only by blocks past the first batch and for
// the operands.
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));
template <typename S, uint32_t kTiles, int kA, int kM, bool kGuarded = false>
__global__ __launch_bounds__(kBlock) void view_tile_vec_kernel(
    const S *__restrict__ x, S *__restrict__ y, uint32_t tiles_l, uint32_t tl_mul,
    uint32_t tl_shift, uint32_t tiles_p, uint32_t tp_mul, uint32_t tp_shift, uint32_t np,
    uint32_t nl, uint32_t xs_last, uint32_t x_offset, uint32_t ys, const S *__restrict__ addend,
    const S *__restrict__ mult, TilePlan plan) {
    static_assert(sizeof(S) == 2 || sizeof(S) == 4, "2- or 4-byte elements");
    constexpr uint32_t E = Vec16<S>::N;              // elements per 16-byte vector
    constexpr uint32_t kSlots = kTile / E;           // vectors per 64-element row
    constexpr uint32_t kRowsPerPass = kBlock / kSlots;
    constexpr uint32_t kPasses = kTile / kRowsPerPass;
    using U = std::conditional_t<sizeof(S) == 2, uint16_t, uint32_t>;
    __shared__ u32x4 tile[kTiles][kTile][kSlots];
    const uint32_t block = blockIdx.x;
    const uint32_t rest = fast_div(block, FastDiv{tiles_l, tl_mul, tl_shift});
    const uint32_t tl = block - rest * tiles_l;
    uint32_t batch = fast_div(rest, FastDiv{tiles_p, tp_mul, tp_shift});
    const uint32_t tp = rest - batch * tiles_p;
    int64_t xb = (int64_t)x_offset;
    uint64_t yb = 0, ab = 0, mb = 0;
    if (batch != 0) {   // block-uniform; batch 0 has every batch index 0
        const BatchBase base(plan, batch);
        xb = base.x;
        yb = base.y;
        ab = base.a;
        mb = base.m;
    }
    const uint32_t p0 = kGuarded ? tp * kTile : min(tp * kTile, np - kTile);
    const uint32_t c = threadIdx.x % kSlots, r0 = threadIdx.x / kSlots;
    // the first index of tile tt along the last dim; tiles past the end repeat
    // the last one (and store nothing)
    auto first_l = [&](uint32_t tt) {
        const uint32_t l = (tl * kTiles + tt) * kTile;
        return kGuarded ? l : min(l, nl - kTile);
    };
#pragma unroll
    for (uint32_t tt = 0; tt < kTiles; ++tt)
#pragma unroll
    for (uint32_t pass = 0; pass < kPasses; ++pass) {
        const uint32_t l = r0 + kRowsPerPass * pass;
        u32x4 v = {0u, 0u, 0u, 0u};
        if (!kGuarded || (first_l(tt) + l < nl && p0 + E * c < np))
            v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_any *>(
                x + xb + (int64_t)(first_l(tt) + l) * xs_last + p0 + E * c));
        tile[tt][l][c ^ (l / E % kSlots)] = v;
    }
    // operands of this lane's output vectors
    Vec16<S> av[kA == kVector ? kTiles * kPasses : 1], mv[kM == kVector ? kTiles * kPasses : 1];
    float as[kA == kScalar ? kPasses : 1], ms[kM == kScalar ? kPasses : 1];
    if constexpr (kA != kNone || kM != kNone) {
        const uint64_t ap = plan.a_stride[plan.p], mp = plan.m_stride[plan.p];
#pragma unroll
        for (uint32_t pass = 0; pass < kPasses; ++pass) {
            const uint64_t pi = p0 + r0 + kRowsPerPass * pass;
            if constexpr (kA == kScalar) as[pass] = Elem<S>::load(addend[ab + pi * ap]);
            if constexpr (kM == kScalar) ms[pass] = Elem<S>::load(mult[mb + pi * mp]);
#pragma unroll
            for (uint32_t tt = 0; tt < kTiles; ++tt) {
                const uint32_t li = first_l(tt) + E * c;
                if constexpr (kA == kVector)
                    av[tt * kPasses + pass] = __builtin_bit_cast(
                        Vec16<S>, (u32x4)*reinterpret_cast<const u32x4_any *>(addend + ab + pi * ap + li));
                if constexpr (kM == kVector)
                    mv[tt * kPasses + pass] = __builtin_bit_cast(
                        Vec16<S>, (u32x4)*reinterpret_cast<const u32x4_any *>(mult + mb + pi * mp + li));
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t tt = 0; tt < kTiles; ++tt)
#pragma unroll
    for (uint32_t pass = 0; pass < kPasses; ++pass) {
        const uint32_t pr = r0 + kRowsPerPass * pass;
        if (kGuarded && (p0 + pr >= np || first_l(tt) + E * c >= nl)) continue;
        // element (l = E c + k, p = pr): row l, slot (pr / E) ^ c, element pr % E
        uint32_t h[E];
#pragma unroll
        for (uint32_t k = 0; k < E; ++k) {
            const U *row = reinterpret_cast<const U *>(&tile[tt][E * c + k][0]);
            h[k] = row[(((pr / E) ^ c) * E) + pr % E];
        }
        u32x4 o;
        if constexpr (sizeof(S) == 2)
            o = u32x4{h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16};
        else
            o = u32x4{h[0], h[1], h[2], h[3]};
        if constexpr (kA != kNone || kM != kNone) {
            Vec16<S> ov = __builtin_bit_cast(Vec16<S>, o);
#pragma unroll
            for (uint32_t k = 0; k < E; ++k) {
                float r = Elem<S>::load(ov.v[k]);
                if constexpr (kA == kVector) r = r + Elem<S>::load(av[tt * kPasses + pass].v[k]);
                if constexpr (kA == kScalar) r = r + as[pass];
                if constexpr (kM == kVector) r = rounded_f32<S>(r * Elem<S>::load(mv[tt * kPasses + pass].v[k]));
                if constexpr (kM == kScalar) r = rounded_f32<S>(r * ms[pass]);
                ov.v[k] = Elem<S>::store(r);
            }
            o = __builtin_bit_cast(u32x4, ov);
        }
        if (kTiles == 1 || kGuarded || (tl * kTiles + tt) * kTile < nl)
            *reinterpret_cast<u32x4_any *>(y + yb + (uint64_t)(p0 + pr) * ys + first_l(tt) + E * c) = o;
    }
}

inline bool aligned16(const void *p) { return p == nullptr || ((uintptr_t)p & 15u) == 0; }

// Gather-path plan for a coalesced view, or false when the view does not fit
// it: innermost dim not contiguous or not whole vectors, offsets not
// vector-aligned, or a plane whose lane offsets or a grid that exceeds 32 bits.
template <typename S>
bool gather_plan(const Coalesced &c, uint64_t x_offset, uint64_t n, bool have_a, bool have_m,
                 GatherPlan *plan, uint32_t *blocks) {
    constexpr uint64_t E = Vec16<S>::N;
    const int last = c.rank - 1;
    if (c.x_stride[last] != 1 || c.shape[last] % E != 0 || x_offset % E != 0) return false;
    for (int d = 0; d < last; ++d)
        if (c.x_stride[d] < 0) return false;  // offsets are unsigned sums
    const bool a_vec = have_a && c.a_stride[last] != 0;
    const bool m_vec = have_m && c.m_stride[last] != 0;
    for (int d = 0; d < last; ++d) {
        if (c.x_stride[d] % E != 0) return false;
        if (a_vec && c.a_stride[d] % E != 0) return false;
        if (m_vec && c.m_stride[d] % E != 0) return false;
    }
    const uint64_t vecs = c.shape[last] / E;
    const uint64_t rows = c.rank >= 2 ? c.shape[last - 1] : 1;
    const uint64_t row_x = c.rank >= 2 ? (uint64_t)c.x_stride[last - 1] : 0;
    const uint64_t row_a = c.rank >= 2 ? c.a_stride[last - 1] : 0;
    const uint64_t row_m = c.rank >= 2 ? c.m_stride[last - 1] : 0;
    const uint64_t plane = rows * vecs;
    const uint64_t plane_blocks = (plane + kBlock - 1) / kBlock;
    const uint64_t outer = n / (plane * E);
    const uint64_t lim = 0xffffffffull;
    if (plane > lim / 2 || plane_blocks * outer > 0x7fffffffull || outer > lim ||
        (rows - 1) * row_x + vecs * E > lim || (rows - 1) * row_a + vecs * E > lim ||
        (rows - 1) * row_m + vecs * E > lim)
        return false;
    *plan = GatherPlan{};
    plan->outer_rank = c.rank >= 2 ? c.rank - 2 : 0;
    for (int d = 0; d < plan->outer_rank; ++d) {
        plan->outer[d] = make_fast_div((uint32_t)c.shape[d]);
        plan->ox[d] = (uint64_t)c.x_stride[d];
        plan->oa[d] = c.a_stride[d];
        plan->om[d] = c.m_stride[d];
    }
    plan->plane_blocks = make_fast_div((uint32_t)plane_blocks);
    plan->vecs = make_fast_div((uint32_t)vecs);
    plan->vecs_log2 = (vecs & (vecs - 1)) == 0 ? __builtin_ctzll(vecs) : -1;
    plan->plane = (uint32_t)plane;
    plan->row_x = (uint32_t)row_x;
    plan->row_a = (uint32_t)row_a;
    plan->row_m = (uint32_t)row_m;
    plan->x_offset = x_offset;
    *blocks = (uint32_t)(plane_blocks * outer);
    return true;
}

// ---- copy path ---------------------------------------------------------------

// A view that coalesces to one contiguous run, with neither operand, is a
// copy of that run: one 16-byte vector per lane over a 1-D grid, the
// arguments plain scalars (preloaded in SGPRs), nothing in front of the load
// but the lane's offset. kWhole: the run is a whole number of blocks, so no
// lane needs the bounds select; otherwise lanes past the end re-read vector
// 0 and the last block's output window ends at the run's end (their stores
// are dropped by the range check). Measured on MI355X against the gather
// kernels' copy of the same run: 0.7-0.8 us less per launch at 67-268 MB
// (the gather kernels form outer coordinates and 64-bit addresses first).
template <typename S, bool kWhole>
__global__ __launch_bounds__(kBlock) void view_copy_kernel(const S *__restrict__ x,
                                                           S *__restrict__ y, uint32_t vecs) {
    constexpr uint32_t E = Vec16<S>::N;
    const uint32_t v0 = blockIdx.x * kBlock;
    const uint32_t v = v0 + threadIdx.x;
    const Vec16<S> xv = load16_stream(x + (size_t)(kWhole || v < vecs ? v : 0u) * E);
    const uint32_t left = vecs - v0;
    const OutWindow w(y + (size_t)v0 * E, (kWhole || left >= kBlock ? kBlock : left) * 16u);
    w.store16(threadIdx.x * 16u, xv);
}

template <typename S>
hipError_t launch_view(const S *x, const k::ViewArgs &v, const S *addend,
                       const S *mult, S *y, hipStream_t s) {
    const int rank = v.rank;
    if (rank < 1 || rank > kMaxRank) return hipErrorInvalidValue;
    uint64_t n = 1;
    for (int d = 0; d < rank; ++d) n *= v.shape[d];
    if (n == 0) return hipSuccess;
    uint64_t a_stride[kMaxRank] = {}, m_stride[kMaxRank] = {};
    broadcast_strides(v.addend_shape, rank, a_stride);
    broadcast_strides(v.mult_shape, rank, m_stride);
    if (!addend) std::fill(a_stride, a_stride + rank, 0);
    if (!mult) std::fill(m_stride, m_stride + rank, 0);
    const Coalesced c = coalesce(v, a_stride, m_stride);
    const int last = c.rank - 1;

    if (!addend && !mult && c.rank == 1 && c.x_stride[0] == 1 && aligned16(x + v.offset) &&
        aligned16(y) && n % Vec16<S>::N == 0 && n / Vec16<S>::N <= 0xffffffffull - kBlock) {
        const uint32_t vecs = (uint32_t)(n / Vec16<S>::N);
        const dim3 grid((vecs + kBlock - 1) / kBlock), block(kBlock);
        if (vecs % kBlock == 0)
            hipLaunchKernelGGL((view_copy_kernel<S, true>), grid, block, 0, s, x + v.offset, y, vecs);
        else
            hipLaunchKernelGGL((view_copy_kernel<S, false>), grid, block, 0, s, x + v.offset, y, vecs);
        return hipGetLastError();
    }

    GatherPlan gp;
    uint32_t blocks = 0;
    if (aligned16(x) && aligned16(y) && aligned16(addend) && aligned16(mult) &&
        gather_plan<S>(c, v.offset, n, addend != nullptr, mult != nullptr, &gp, &blocks)) {
        const int ka = !addend ? kNone : c.a_stride[last] != 0 ? kVector : kScalar;
        const int km = !mult ? kNone : c.m_stride[last] != 0 ? kVector : kScalar;
        ShortPlan sp;
        dim3 short_grid;
        const bool use_short = short_plan<S>(c, v.offset, n, &sp, &short_grid);
        const dim3 grid(blocks), block(kBlock);
#define ICSDK_GATHER(A, M)                                                                      \
    do {                                                                                        \
        if (use_short)                                                                          \
            hipLaunchKernelGGL((view_gather_short_kernel<S, A, M>), short_grid, block, 0, s, x,  \
                               addend, mult, y, sp);                                            \
        else                                                                                    \
            hipLaunchKernelGGL((view_gather_kernel<S, A, M>), grid, block, 0, s, x, addend,     \
                               mult, y, gp);                                                    \
    } while (0)
        switch (ka * 3 + km) {
            case 0: ICSDK_GATHER(kNone, kNone); break;
            case 1: ICSDK_GATHER(kNone, kVector); break;
            case 2: ICSDK_GATHER(kNone, kScalar); break;
            case 3: ICSDK_GATHER(kVector, kNone); break;
            case 4: ICSDK_GATHER(kVector, kVector); break;
            case 5: ICSDK_GATHER(kVector, kScalar); break;
            case 6: ICSDK_GATHER(kScalar, kNone); break;
            case 7: ICSDK_GATHER(kScalar, kVector); break;
            default: ICSDK_GATHER(kScalar, kScalar); break;
        }
#undef ICSDK_GATHER
        return hipGetLastError();
    }

    // tile path: exactly one coalesced dim p != last has x stride 1
    int p = -1;
    for (int d = 0; d < last; ++d)
        if (c.x_stride[d] == 1) p = p < 0 ? d : -2;
    if (p >= 0 && c.x_stride[last] != 1) {
        TilePlan plan{};
        plan.rank = c.rank;
        plan.p = p;
        uint64_t ys = 1;
        for (int d = last; d >= 0; --d) {
            plan.shape[d] = c.shape[d];
            plan.x_stride[d] = c.x_stride[d];
            plan.a_stride[d] = c.a_stride[d];
            plan.m_stride[d] = c.m_stride[d];
            plan.y_stride[d] = ys;
            ys *= c.shape[d];
        }
        plan.x_offset = v.offset;
        plan.batches = n / (c.shape[p] * c.shape[last]);
        const uint64_t np = c.shape[p], nl = c.shape[last], lim = 0xffffffffull;
        const int ka = !addend ? kNone : c.a_stride[last] != 0 ? kVector : kScalar;
        const int km = !mult ? kNone : c.m_stride[last] != 0 ? kVector : kScalar;
        // 64 x 64 tiles of vectors (the scalar arguments hold dims, the x row
        // stride, the offset and the output row stride in 32 bits; the
        // operands' rows run along last)
        const bool fits32 = np + kTile <= lim && nl + 4 * kTile <= lim && c.x_stride[last] > 0 &&
                            (uint64_t)c.x_stride[last] <= lim && v.offset <= lim && plan.y_stride[p] <= lim;
        // An operand that is the output (y = view(x) + y) is read by the lane
        // that writes its element; a tile that overlaps another one would
        // read what that one has written.
        const bool both = np >= kTile && nl >= kTile;
        const bool overlap = np % kTile != 0 || nl % kTile != 0;
        const bool in_place = (addend && addend == y) || (mult && mult == y);
        // whole aligned vectors in every x row, batch offset and output row
        constexpr uint64_t E = Vec16<S>::N;
        constexpr uint32_t kGuardedTiles = sizeof(S) == 2 ? 4 : 1;
        bool whole = !addend && !mult && np % E == 0 && nl % E == 0 && v.offset % E == 0 && aligned16(x) &&
                     aligned16(y);
        for (int d = 0; d <= last; ++d)
            if (d != p && c.x_stride[d] % (int64_t)E != 0) whole = false;
        // With a dim below 64 the bounds-tested form, where a block still moves
        // enough: views that one tile holds from 400 elements (us at 6.3 M
        // elements in batches, here / adaptive tiles / one element per lane: f16
        // 32 x 32 11.9 / 13.1 / 25, 48 x 48 8.7 / 14.1 / 25, f32 20 x 20 21.7 /
        // 26.6 / 24.5; f32 from 256, 16 x 16 26.7 / 39 / 25.4), longer ones from 1280
        // per block (f16 32 x 1000 10.0 / 12.3 / 26, 512 x 16 12.5 / 11.0 / 26, 504 x 8
        // 26 / 12 / 25; f32 1000 x 32 11.3 / 12.3 / 25.5, 500 x 4 29 / 16 / 25), f32 with
        // a short p from 2560 (40 x 1000 13.4 / 14.1 / 36, 32 x 1000 13.9 / 12.5 / 34). With
        // both dims of 64 f32 takes it where more than one tile in 16 would
        // overlap another one (overlapping / here, us: 12580 x 500 14.1 / 12.2,
        // 92000 x 68 15.8 / 11.3; but 4096 x 4000 20.1 / 22.7, 3000 x 3000 16.5 /
        // 17.1), and from 1025 to 2048 tiles, the second half of the one round
        // that the CUs hold of either form: it wins at every shape measured there
        // (2000 x 2560 8.3 / 7.1, 512 x 12288 9.1 / 8.1, 2688 x 2688 10.5 / 9.3; 1024
        // tiles 5.3 / 5.5, 2500 14.3 / 15.2).
        const uint64_t moved = std::min<uint64_t>(np, kTile) * std::min<uint64_t>(nl, kTile * kGuardedTiles);
        const uint64_t tiles_p = (np + kTile - 1) / kTile, tiles_l = (nl + kTile - 1) / kTile;
        const bool ragged = 16 * ((np % kTile != 0) * tiles_l + (nl % kTile != 0) * tiles_p) > tiles_p * tiles_l;
        const uint64_t all_tiles = plan.batches * tiles_p * tiles_l;
        const bool half_round = all_tiles > 1024 && all_tiles <= 2048;
        constexpr bool f16 = sizeof(S) == 2;
        const bool one_tile = np <= kTile && nl <= kTile && np * nl >= (f16 ? 400 : 256);
        const bool guarded = whole && (both ? f16 || ragged || half_round
                                            : one_tile || moved >= (!f16 && np < kTile ? 2560 : 1280));
        if (fits32 && (guarded || (both && !(in_place && overlap) && c.a_stride[last] <= 1 && c.m_stride[last] <= 1))) {
            plan.tiles_p = (uint32_t)tiles_p;
            const uint32_t per = guarded ? kGuardedTiles : sizeof(S) == 2 && all_tiles >= 2048 && nl > kTile ? 2 : 1;
            const uint32_t spans_l = (uint32_t)((nl + per * kTile - 1) / (per * kTile));
            const uint64_t vblocks = plan.batches * plan.tiles_p * spans_l;
            if (vblocks < (uint64_t{1} << 24)) {
                const FastDiv dl = make_fast_div(spans_l), dp = make_fast_div(plan.tiles_p);
                auto go = [&](auto kernel) {
                    hipLaunchKernelGGL(kernel, dim3((unsigned)vblocks), dim3(kBlock), 0, s, x, y, spans_l,
                                       dl.multiplier, dl.shift, plan.tiles_p, dp.multiplier, dp.shift,
                                       (uint32_t)np, (uint32_t)nl, (uint32_t)c.x_stride[last],
                                       (uint32_t)v.offset, (uint32_t)plan.y_stride[p], addend, mult, plan);
                    return hipGetLastError();
                };
#define ICSDK_TILE_VEC(A, M)                                                                     \
    do {                                                                                         \
        if constexpr (sizeof(S) == 2)                                                            \
            if (per == 2) return go(view_tile_vec_kernel<S, 2, A, M>);                           \
        return go(view_tile_vec_kernel<S, 1, A, M>);                                             \
    } while (0)
                if (guarded) return go(view_tile_vec_kernel<S, kGuardedTiles, kNone, kNone, true>);
                switch (ka * 3 + km) {
                    case 0: ICSDK_TILE_VEC(kNone, kNone);
                    case 1: ICSDK_TILE_VEC(kNone, kVector);
                    case 2: ICSDK_TILE_VEC(kNone, kScalar);
                    case 3: ICSDK_TILE_VEC(kVector, kNone);
                    case 4: ICSDK_TILE_VEC(kVector, kVector);
                    case 5: ICSDK_TILE_VEC(kVector, kScalar);
                    case 6: ICSDK_TILE_VEC(kScalar, kNone);
                    case 7: ICSDK_TILE_VEC(kScalar, kVector);
                    default: ICSDK_TILE_VEC(kScalar, kScalar);
                }
#undef ICSDK_TILE_VEC
            }
        }
        // Adaptive tiles: the shorter dim whole up to 64 (32 for small tiles),
        // the other one as long as fits the tile. Small ones where that makes
        // more, shorter blocks (views of fewer than 1024 large tiles), and where
        // the large ones are mostly empty: up to twice as many small ones cost less
        // (us, f16 at 6.3 M elements, large / small: 24 x 24, one tile either way, 36 /
        // 20, 4 x 500 15.5 / 13.5, 8 x 500 11.8 / 13.5). A block is paid whether
        // its tile is full or not (1.5 to 2.5 ns of the launch): tiles of fewer than
        // 512 elements go to one element per lane, 4 ns per 1000 elements (us,
        // here / there: 2 x 3 1530 / 25, 16 x 16 39 / 25, 16 x 32 21 / 25; with
        // operands 2137 / 28, 55 / 28, 30 / 29).
        uint64_t ep = 0, el = 0;
        auto cut = [&](uint64_t elems, uint64_t side) {
            ep = std::min(np, side), el = std::min(nl, side);
            if (np <= nl) el = std::min(nl, std::max<uint64_t>(elems / ep / side, 1) * side);
            else ep = std::min(np, std::max<uint64_t>(elems / el / side, 1) * side);
            return plan.batches * ((np + ep - 1) / ep) * ((nl + el - 1) / el);
        };
        const uint64_t large_blocks = cut(kTileElems, 64), small_blocks = cut(kTileElemsSmall, 32);
        const bool small = n <= 1024ull * kTileElems || small_blocks <= 2 * large_blocks;
        const uint64_t elems = small ? kTileElemsSmall : kTileElems;
        const uint64_t blocks = cut(elems, small ? 32 : 64);
        plan.tile_p = make_fast_div((uint32_t)ep);
        plan.tile_l = make_fast_div((uint32_t)el);
        plan.tiles_p = (uint32_t)((np + ep - 1) / ep);
        plan.tiles_l = (uint32_t)((nl + el - 1) / el);
        if (blocks < (uint64_t{1} << 24) && (n / blocks >= 480 || blocks <= 1024) && ep * el <= elems && (ep | 1u) * el <= elems / 2 * 3) {
            auto go = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(kBlock), 0, s, x, addend, mult, y, plan);
                return hipGetLastError();
            };
#define ICSDK_TILE(A, M)                                                                           \
    return small ? go(view_tile_kernel<S, kTileElemsSmall, A, M>) : go(view_tile_kernel<S, kTileElems, A, M>)
            if (addend && mult) ICSDK_TILE(true, true);
            if (addend) ICSDK_TILE(true, false);
            if (mult) ICSDK_TILE(false, true);
            ICSDK_TILE(false, false);
#undef ICSDK_TILE
        }
    }

    ScalarPlan plan{};
    plan.rank = c.rank;
    for (int d = 0; d < c.rank; ++d) {
        plan.shape[d] = c.shape[d];
        plan.x_stride[d] = c.x_stride[d];
        plan.a_stride[d] = c.a_stride[d];
        plan.m_stride[d] = c.m_stride[d];
    }
    plan.x_offset = v.offset;
    uint64_t grid = (n + kBlock * 4 - 1) / (kBlock * 4);
    if (grid > (1u << 20)) grid = 1u << 20;
    hipLaunchKernelGGL((view_scalar_kernel<S>), dim3((unsigned)grid), dim3(kBlock), 0, s, x,
                       addend, mult, y, (size_t)n, plan);
    return hipGetLastError();
}

}  // namespace

namespace k {

hipError_t view_add_mul_f32(const float *x, const ViewArgs &v, const float *addend,
                            const float *mult, float *y, hipStream_t s) {
    return launch_view<float>(x, v, addend, mult, y, s);
}

hipError_t view_add_mul_f16(const uint16_t *x, const ViewArgs &v, const uint16_t *addend,
                            const uint16_t *mult, uint16_t *y, hipStream_t s) {
    return launch_view<_Float16>(reinterpret_cast<const _Float16 *>(x), v,
                                 reinterpret_cast<const _Float16 *>(addend),
                                 reinterpret_cast<const _Float16 *>(mult),
                                 reinterpret_cast<_Float16 *>(y), s);
}

}  // namespace k
}  // namespace icsdk
