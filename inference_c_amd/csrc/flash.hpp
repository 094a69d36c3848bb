// MFMA flash attention kernels (f16 and f32), shared by the translation units
// that instantiate them: k_attention.hip (head dims 64 and 128) and
// k_attention_dims.hip (every other head dim up to 256).
#pragma once

#include "kern_common.hpp"
#include "kernels.hpp"

namespace icsdk {
namespace flash {

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
// mask rows start at any element
typedef uint32_t u32x4_2 __attribute__((ext_vector_type(4), aligned(2)));
typedef float f32x4_4 __attribute__((ext_vector_type(4), aligned(4)));

struct SdpaArgs {
    uint32_t batch, qh, kvh, group;   // group = qh / kvh
    uint32_t ql, kl, dim, vdim;
    uint32_t causal_offset;           // kl > ql ? kl - ql : 0
    float scale;
    int causal;
    // Flash work schedule. Every (batch, head) has `items` work items; item r
    // is key-tile part `part` of `parts` of query block `qblock`, packed as
    // qblock | part << 16 | parts << 24 in item[r] when `table` is set (else
    // item r is query block qblocks - 1 - r, whole). A query block of n key
    // tiles has split_parts(n, split_tiles) parts; a part's block writes its
    // unnormalised output rows to part_o[part][row][D] and {running max, sum,
    // NaN flag, 0} to part_ml[part][row], merged by sdpa_combine_kernel.
    uint32_t items, qblocks;
    uint32_t split_tiles;   // 0: no query block is split
    uint32_t table;
    uint32_t xcd_heads;     // keep the q-heads of one kv head on one XCD
    float *part_o;
    f32x4 *part_ml;
    uint32_t item[128];
};
constexpr uint32_t kMaxFlashItems = 128;
constexpr uint32_t kMaxKeyParts = 8;
constexpr uint32_t kMinPartTiles = 4;   // a part amortises its set-up and the merge

// Key tiles (of tk keys) that the queries of query block j (bm queries) may
// see: all kl keys, or when causal those up to its last query + offset.
__host__ __device__ inline uint32_t flash_tiles(uint32_t ql, uint32_t kl, bool causal,
                                                uint32_t offset, uint32_t bm, uint32_t tk,
                                                uint32_t j) {
    const uint32_t last = j * bm + bm - 1 < ql - 1 ? j * bm + bm - 1 : ql - 1;
    const uint64_t seen = (uint64_t)last + offset + 1;
    const uint64_t key_end = causal && seen < kl ? seen : kl;
    return (uint32_t)((key_end + tk - 1) / tk);
}

// Parts of a query block of `tiles` key tiles: about tiles / split_tiles,
// each of at least kMinPartTiles tiles, at most kMaxKeyParts.
__host__ __device__ inline uint32_t split_parts(uint32_t tiles, uint32_t split_tiles) {
    if (split_tiles == 0) return 1;
    uint32_t n = (tiles + split_tiles - 1) / split_tiles;
    const uint32_t most = tiles / kMinPartTiles;
    n = n < most ? n : most;
    n = n < kMaxKeyParts ? n : kMaxKeyParts;
    return n < 1 ? 1 : n;
}

// ---- row kernel ----------------------------------------------------------------

constexpr int kMaxRowRegs = 8;  // D, Dv <= 8 * 64

__device__ inline float broadcast_lane(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// exp for the softmax weights: libm-accurate for f32 outputs, the hardware
// exp2 path for f16 outputs (its error is far below half an f16 ulp).
template <typename S>
__device__ inline float attn_exp(float x) {
    if constexpr (sizeof(S) == 2) return fast_exp(x);
    else return expf(x);
}

// Score of the lane's key row: q . k in d order (sequential f32 sums, no
// contraction), q[d] taken from lane d % 64 of register d / 64. kVec: rows
// are whole, aligned 16-byte vectors.
template <typename S, bool kVec>
__device__ inline float row_dot(const float (&qreg)[kMaxRowRegs], const S *krow, uint32_t dim) {
    constexpr uint32_t E = Vec16<S>::N;
    float sum = 0.0f;
#pragma unroll
    for (int t = 0; t < kMaxRowRegs; ++t) {
        const uint32_t d0 = (uint32_t)t * kWave;
        if (d0 >= dim) break;
        const uint32_t dn = min(dim - d0, (uint32_t)kWave);
        if constexpr (kVec) {
            for (uint32_t dd = 0; dd < dn; dd += E) {
                const Vec16<S> kv = load16(krow + d0 + dd);
#pragma unroll
                for (uint32_t e = 0; e < E; ++e)
                    sum = sum + broadcast_lane(qreg[t], (int)(dd + e)) * Elem<S>::load(kv.v[e]);
            }
        } else {
            for (uint32_t dd = 0; dd < dn; ++dd)
                sum = sum + broadcast_lane(qreg[t], (int)dd) * Elem<S>::load(krow[d0 + dd]);
        }
    }
    return sum;
}

// One query row by one wave (the row kernel; the header comment of
// k_attention.hip describes it).
template <typename S, bool kVec>
__device__ inline void sdpa_row(const S *__restrict__ q, const S *__restrict__ k,
                                const S *__restrict__ v, const S *__restrict__ mask,
                                S *__restrict__ out, const SdpaArgs &a, size_t row,
                                uint32_t lane) {
    const uint32_t i = (uint32_t)(row % a.ql);          // query position
    const size_t bh = row / a.ql;                        // batch * qh + head
    const uint32_t head = (uint32_t)(bh % a.qh);
    const size_t b = bh / a.qh;
    const size_t kv = b * a.kvh + head / a.group;
    const S *qrow = q + row * a.dim;
    const S *kbase = k + kv * a.kl * a.dim;
    const S *vbase = v + kv * a.kl * a.vdim;

    // q[d] lives in lane d % 64, register d / 64
    float qreg[kMaxRowRegs];
#pragma unroll
    for (int t = 0; t < kMaxRowRegs; ++t) {
        const uint32_t d = lane + t * kWave;
        qreg[t] = d < a.dim ? Elem<S>::load(qrow[d]) : 0.0f;
    }
    float acc[kMaxRowRegs];
#pragma unroll
    for (int t = 0; t < kMaxRowRegs; ++t) acc[t] = 0.0f;
    const float neg_inf = -__builtin_inff();
    float m = neg_inf, l = 0.0f;
    bool nan_seen = false;
    // keys past `last` are masked by the causal rule for this row
    const uint64_t last = a.causal ? (uint64_t)i + a.causal_offset : (uint64_t)a.kl - 1;
    for (uint32_t c0 = 0; c0 < a.kl && (uint64_t)c0 <= last; c0 += kWave) {
        const uint32_t j = c0 + lane;
        const bool live = j < a.kl;
        float s = neg_inf;
        if (live) {
            s = row_dot<S, kVec>(qreg, kbase + (size_t)j * a.dim, a.dim) * a.scale;
            if (mask) s = s + Elem<S>::load(mask[(size_t)i * a.kl + j]);
            if (a.causal && (uint64_t)j > last) s = neg_inf;
        }
        // a NaN score never becomes the max, but a row with a finite max and
        // a NaN score is NaN (its sum is)
        nan_seen = nan_seen || wave_any(s != s);
        const float m_new = fmaxf(m, wave_max(s));
        if (m_new == neg_inf) continue;                  // nothing visible yet
        const float alpha = attn_exp<S>(m - m_new);      // 0 when m was -inf
        const float p = live ? attn_exp<S>(s - m_new) : 0.0f;
        l = l * alpha + wave_sum(p);
        m = m_new;
        const uint32_t n = min(a.kl - c0, (uint32_t)kWave);
#pragma unroll
        for (int t = 0; t < kMaxRowRegs; ++t) acc[t] = acc[t] * alpha;
        for (uint32_t jj = 0; jj < n; ++jj) {
            const float pj = broadcast_lane(p, (int)jj);
            const S *vrow = vbase + (size_t)(c0 + jj) * a.vdim;
#pragma unroll
            for (int t = 0; t < kMaxRowRegs; ++t) {
                const uint32_t e = lane + t * kWave;
                if (e < a.vdim) acc[t] = acc[t] + pj * Elem<S>::load(vrow[e]);
            }
        }
    }
    const bool zero = !__builtin_isfinite(m);
    const float inverse = l == 0.0f ? 0.0f : 1.0f / l;
    const float nan = __builtin_nanf("");
    S *orow = out + row * a.vdim;
#pragma unroll
    for (int t = 0; t < kMaxRowRegs; ++t) {
        const uint32_t e = lane + t * kWave;
        if (e < a.vdim)
            orow[e] = Elem<S>::store(zero ? 0.0f : nan_seen ? nan : acc[t] * inverse);
    }
}

// ---- MFMA flash kernels ---------------------------------------------------------

// kAnyDim kernels: D is the padded head dim (at least a.dim and a.vdim, both
// a whole number of 16-byte vectors); rows are a.dim and a.vdim wide in
// memory, Q and K columns past a.dim are zeros, and output columns past
// a.vdim are not stored. Without it the kernel's head dim is exactly D.

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));

// A block owns BM queries of one (batch, head): 32 per wave (KS waves per
// 32 queries when the key tiles are split between them). Keys come in tiles
// of 64, staged in LDS by the whole block, double-buffered: the next step's
// global loads are issued before the current step is computed and land in
// the other buffer afterwards, so one barrier per step separates the
// writers of a buffer from its readers. K and V are both stored as
// [key][dim] rows, as they are in memory (16-byte loads and stores, 256
// contiguous bytes per row at D 128).
//
// v_mfma_f32_32x32x16_f16 lane layout (checked on the device): A[m][k] in
// lane l at m = l % 32, k = 8 (l / 32) + i; B[k][n] at n = l % 32,
// k = 8 (l / 32) + i; D[m][n] at n = l % 32, m = 8 (r / 4) + 4 (l / 32) + r % 4.
//
// Scores: S^T = K Q^T per 32-key half tile (A = K rows from LDS, B = the
// wave's Q rows, loaded once), so lane l holds query l % 32 and, of each
// half tile, keys 8 (r / 4) + 4 (l / 32) + r % 4; lane l ^ 32 holds the rest.
// The online softmax runs per lane pair (one swizzle for the max, one for
// the sum). P^T is then already the B operand of out^T = V^T P^T: chunk c of
// its k dimension is p[8c .. 8c + 7], keys 16c + 8 (i / 4) + 4 (l / 32) + i % 4.
// The matching A fragment (V^T: lane l needs V[16c + 4h + k][d] and
// V[16c + 8 + 4h + k][d], k = 0..3, d = l % 32, h = l / 32) comes from the
// [key][dim] V rows through two ds_read_b64_tr_b16: within each 16-lane
// group that instruction hands lane j element j % 4 of the 4-element vectors
// addressed by lanes j / 4 + 4k, k = 0..3 (checked on the device), so lane
// i of group g addresses row 16c + 4 (g / 2) + i / 4 (+ 8), columns
// 16 (g % 2) + 4 (i % 4) .. + 3.
constexpr int kFlashN = 64;    // keys per tile
constexpr float kLazyLog2 = 8.0f;   // rescale when a row maximum grows by more than 2^8
// s_waitcnt vmcnt(0) (GFX9 encoding: expcnt and lgkmcnt at their no-wait maxima)
constexpr int kWaitVmcnt0 = 0x0F70;

// Block -> work item. Blocks are numbered item-rank-major (all (batch, head)
// pairs of the largest item first), so the blocks dispatched first are the
// longest and the short ones fill in behind them. MI355X dispatches a
// launch's workgroups to its 8 XCDs round-robin (block b on XCD b % 8) and
// each XCD has its own 4 MB L2: with xcd_heads (batch * kv heads divisible
// by 8, so b % 8 == p % 8), XCD x takes the q-heads of kv units x, x + 8, ...
// and a kv head's K/V tiles are fetched into one L2 instead of all eight.
struct FlashItem {
    uint32_t bh, qblock, part, parts;
};
__device__ inline FlashItem flash_item(const SdpaArgs &a, uint32_t block) {
    const uint32_t bhs = a.batch * a.qh;
    const uint32_t r = block / bhs, p = block % bhs;
    FlashItem it;
    if (a.xcd_heads) {
        const uint32_t x = p % 8, i = p / 8;
        it.bh = (x + 8 * (i / a.group)) * a.group + i % a.group;
    } else {
        it.bh = p;
    }
    if (a.table) {
        const uint32_t e = a.item[r];
        it.qblock = e & 0xffffu;
        it.part = (e >> 16) & 0xffu;
        it.parts = e >> 24;
    } else {
        it.qblock = a.qblocks - 1 - r;
        it.part = 0;
        it.parts = 1;
    }
    return it;
}

// Max and sum of a value over the lane pair (l, l ^ 32). v_permlane32_swap
// with both operands v leaves every lane holding its own value in one result
// and its partner's in the other (lanes 0-31 keep r0 and receive lane + 32 in
// r1; lanes 32-63 receive lane - 32 in r0 and keep r1), so one cross-lane
// VALU op replaces a round trip through LDS (ds_bpermute).
// The two halves of the wave swap values with v_permlane32_swap: each lane
// gets back its own value and the one of lane +-32. The vector's elements
// are copied into scalars before the bit cast (a bit cast of an element of
// the returned vector reads element 0).
__device__ inline float pair_value(float v, float &partner) {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const unsigned lo = r[0], hi = r[1];
    partner = __builtin_bit_cast(float, hi);
    return __builtin_bit_cast(float, lo);
}
__device__ inline float pair_max(float v) {
    float b;
    const float a = pair_value(v, b);
    return fmaxf(a, b);
}
__device__ inline float pair_sum(float v) {
    float b;
    const float a = pair_value(v, b);
    return a + b;
}

// Scheduling of an unrolled chain of N (LDS read, MFMA) pairs: the first
// kAhead reads, then one MFMA and one read alternately, then the last MFMAs.
// Each MFMA then consumes a fragment read kAhead MFMAs earlier (~128
// cycles), which covers the LDS latency; left to itself the scheduler reads
// one fragment ahead and every MFMA waits for its read.
// (R LDS reads per M MFMAs.)
template <int N, int R = 1, int M = 1>
__device__ inline void lds_read_ahead() {
    constexpr int kAhead = 4;
    constexpr int kMfma = 0x008, kDsRead = 0x100;
    __builtin_amdgcn_sched_group_barrier(kDsRead, kAhead * R, 0);
#pragma unroll
    for (int i = 0; i < N - kAhead; ++i) {
        __builtin_amdgcn_sched_group_barrier(kMfma, M, 0);
        __builtin_amdgcn_sched_group_barrier(kDsRead, R, 0);
    }
    __builtin_amdgcn_sched_group_barrier(kMfma, kAhead * M, 0);
}

// A wave issuing a chain of MFMAs runs at raised priority, so that the
// other waves of its SIMD (in their softmax) take the issue cycles between
// its MFMAs instead of both waves reaching the same phase together.
__device__ inline void mfma_phase_begin() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    __builtin_amdgcn_sched_barrier(0);
}
__device__ inline void mfma_phase_end() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
}

typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef short short4v __attribute__((ext_vector_type(4)));

// Four halves through the LDS transpose read (lane layout above).
__device__ inline half4 lds_read_tr(const _Float16 *p) {
    const short4v r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4v *)(p));
    return __builtin_bit_cast(half4, r);
}

// A split block's result for one query: its lane pair holds the query's
// unnormalised output rows (out^T accumulator layout), the running max and
// sum, and the NaN flag.
template <int VT, bool kAnyDim>
__device__ inline void write_partial(const SdpaArgs &a, uint32_t split, size_t row, uint32_t half,
                                     const float16v (&o)[VT], float m, float l, bool nan_seen) {
    const size_t rows = (size_t)a.batch * a.qh * a.ql;
    float *prow = a.part_o + ((size_t)split * rows + row) * a.vdim;
#pragma unroll
    for (int tt = 0; tt < VT; ++tt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (kAnyDim && 32 * tt + 8 * g + 4 * half >= a.vdim) continue;
            const f32x4 quad = {o[tt][4 * g], o[tt][4 * g + 1], o[tt][4 * g + 2], o[tt][4 * g + 3]};
            *reinterpret_cast<f32x4 *>(prow + 32 * tt + 8 * g + 4 * half) = quad;
        }
    if (half == 0) a.part_ml[(size_t)split * rows + row] = f32x4{m, l, nan_seen ? 1.0f : 0.0f, 0.0f};
}

// Merges the parts of each split query row (rows first_row .. ql - 1 of
// every (batch, head): split query blocks are a suffix, since a later query
// block never sees fewer keys): M = max of the parts' maxima; a row whose M
// is not finite is zero; a NaN flag with a finite M makes the row NaN;
// otherwise out = (sum_s w_s o_s) * (1 / sum_s w_s l_s) with w_s =
// exp(m_s - M) (exp2 when the maxima are in log2 units). One thread per 8
// output elements; kAnyDim: the last group of a row may hold only 4 (an f32
// value dim of 4 mod 8), and an f16 row takes a power of two of lanes, so that
// it lies in one wave: the wave that does a row again stores all of it, and
// no other wave may have a part of the same row to store. (The spare lanes
// of 72 .. 96 wide rows: 16 lanes for 9 .. 12 groups.)
//
// kParts >= the launch's largest part count: every part's (m, l) and output
// vectors are requested up front, unconditionally (a part index past the
// row's own count reads its last part again, which stays in bounds, and is
// left out of the sums), so a row costs one memory round trip; walking the
// parts in a run-time loop waited for each part's loads in turn.
template <typename S, bool kAnyDim> __host__ __device__ inline uint32_t combine_lanes(uint32_t vdim) {
    const uint32_t groups = (vdim + 7) / 8;
    if (!(kAnyDim && sizeof(S) == 2)) return groups;
    uint32_t lanes = 1;
    while (lanes < groups) lanes *= 2;
    return lanes;   // at most 32 (value dims up to 256)
}

template <typename S, bool kLog2, int kParts, bool kAnyDim>
__global__ __launch_bounds__(kBlock) void sdpa_combine_kernel(SdpaArgs a, S *__restrict__ out,
                                                              uint32_t bm, uint32_t tk,
                                                              uint32_t first_row, const S *q,
                                                              const S *k, const S *v,
                                                              const S *mask) {
    const size_t rows = (size_t)a.batch * a.qh * a.ql;
    const uint32_t suffix = a.ql - first_row;
    const uint32_t groups = (a.vdim + 7) / 8, lanes = combine_lanes<S, kAnyDim>(a.vdim);
    const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    const size_t last = (size_t)a.batch * a.qh * suffix * lanes - 1;
    const uint32_t lane_g = (uint32_t)(min(i, last) % lanes);
    const bool live = i <= last && lane_g < groups;
    if (!(kAnyDim && sizeof(S) == 2) && !live) return;   // (the redo below takes whole waves)
    const size_t srow = min(i, last) / lanes;
    const uint32_t g = min(lane_g, groups - 1);
    const uint32_t qi = first_row + (uint32_t)(srow % suffix);
    const size_t row = srow / suffix * a.ql + qi;
    const uint32_t splits = split_parts(
        flash_tiles(a.ql, a.kl, a.causal != 0, a.causal_offset, bm, tk, qi / bm), a.split_tiles);
    f32x4 ml[kParts], po_lo[kParts], po_hi[kParts];
#pragma unroll
    for (int s = 0; s < kParts; ++s) {
        const size_t part = (size_t)min((uint32_t)s, splits - 1) * rows + row;
        ml[s] = a.part_ml[part];
        const f32x4 *po = reinterpret_cast<const f32x4 *>(a.part_o + part * a.vdim + 8 * g);
        po_lo[s] = po[0];
        po_hi[s] = kAnyDim && 8 * g + 4 >= a.vdim ? po[0] : po[1];
    }
    float big = -__builtin_inff();
    bool nan_flag = false;
#pragma unroll
    for (int s = 0; s < kParts; ++s) {
        if ((uint32_t)s < splits) {
            big = fmaxf(big, ml[s].x);
            nan_flag = nan_flag || ml[s].z != 0.0f;
        }
    }
    f32x4 lo = {0.0f, 0.0f, 0.0f, 0.0f}, hi = lo;
    float total = 0.0f;
    if (__builtin_isfinite(big)) {
#pragma unroll
        for (int s = 0; s < kParts; ++s) {
            if ((uint32_t)s >= splits) continue;
            // a part that saw no visible key has sum 0 and output 0; every
            // other part is added even at weight 0, so a NaN it holds stays
            const float w = ml[s].x == -__builtin_inff() ? 0.0f
                            : kLog2 ? __builtin_amdgcn_exp2f(ml[s].x - big) : expf(ml[s].x - big);
            total += w * ml[s].y;
            lo += w * po_lo[s];
            hi += w * po_hi[s];
        }
    }
    const bool zero = !__builtin_isfinite(big);
    const float inverse = total == 0.0f ? 0.0f : 1.0f / total;
    const float nan = __builtin_nanf("");
    S res[8] __attribute__((aligned(16)));
#pragma unroll
    for (int j = 0; j < 8; ++j)
        res[j] = (S)(zero ? 0.0f : nan_flag ? nan : (j < 4 ? lo[j] : hi[j - 4]) * inverse);
    S *orow = out + row * a.vdim + 8 * g;
    if constexpr (sizeof(S) == 2) {
        if (live) *reinterpret_cast<u32x4 *>(orow) = *reinterpret_cast<const u32x4 *>(res);
        if constexpr (kAnyDim) {
            // rows with a finite sum and an output that is not finite are done
            // again by the row routine (see the flash kernel's end)
            float finite = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) finite = __builtin_fmaf(0.0f, lo[j], __builtin_fmaf(0.0f, hi[j], finite));
            uint64_t redo = __builtin_amdgcn_ballot_w64(live && !zero && !nan_flag && finite != 0.0f &&
                                                        __builtin_isfinite(total));
            if (redo != 0) __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);   // the stores above come first
            size_t done = ~size_t{0};
#pragma unroll 1
            while (redo != 0) {
                const int src = __builtin_ctzll(redo);
                redo &= redo - 1;
                const size_t r = (size_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)row, src) |
                                 (size_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(row >> 32), src) << 32;
                if (r != done) sdpa_row<S, true>(q, k, v, mask, out, a, r, threadIdx.x & (kWave - 1));
                done = r;
            }
        }
    } else {
        reinterpret_cast<u32x4 *>(orow)[0] = reinterpret_cast<const u32x4 *>(res)[0];
        if (!kAnyDim || 8 * g + 4 < a.vdim) reinterpret_cast<u32x4 *>(orow)[1] = reinterpret_cast<const u32x4 *>(res)[1];
    }
}

template <int D, int BM, bool kMask, bool kSplit, int KS, bool kAnyDim = false>
__global__ __launch_bounds__(BM * 2 * KS) void sdpa_flash_kernel(const _Float16 *__restrict__ q,
                                                            const _Float16 *__restrict__ k,
                                                            const _Float16 *__restrict__ v,
                                                            const _Float16 *__restrict__ mask,
                                                            _Float16 *__restrict__ out,
                                                            SdpaArgs a) {
    constexpr int QW = BM / 32;              // query groups of 32: one wave each per key part
    constexpr int THREADS = BM * 2 * KS;
    constexpr int KC = D / 16;               // 16-dim chunks of Q K^T
    constexpr int VT = (D + 31) / 32;        // 32-row tiles of out^T
    constexpr int KROW = D + 8;              // LDS row of K (halves)
    // LDS row of V (halves): at least the 32 VT columns the transpose reads
    // touch and 16 or 48 dwords past a multiple of 64, so the 4 rows a
    // transpose read takes per half wave start 16 banks apart
    // (conflict-free)
    constexpr int VROW = VT % 2 ? 32 * VT : 32 * VT + 32;
    static_assert(D % 16 == 0 && VROW / 2 % 32 == 16, "V rows 16 banks apart");
    constexpr int KTILE = kFlashN * KROW;    // LDS halves of one K tile
    constexpr int VTILE = kFlashN * VROW;    // LDS halves of one V tile
    constexpr int TV = kFlashN * D / 8;      // 16-byte vectors per K or V tile
    constexpr int VECS = KS * TV;            // per operand and step (KS tiles)
    constexpr int PER = (VECS + THREADS - 1) / THREADS;   // per thread, per step, per operand
    constexpr bool kWholeLoads = VECS % THREADS == 0;
    static_assert(kWholeLoads || kAnyDim, "tile load split");
    constexpr int RV = D / 8;                // 16-byte vectors per LDS row
    __shared__ __attribute__((aligned(16))) _Float16 tiles_lds[2 * KS * (KTILE + VTILE)];
    _Float16 (*const ks)[KS * KTILE] = reinterpret_cast<_Float16 (*)[KS * KTILE]>(tiles_lds);
    _Float16 (*const vs)[KS * VTILE] =
        reinterpret_cast<_Float16 (*)[KS * VTILE]>(tiles_lds + 2 * KS * KTILE);
    const uint32_t dim = kAnyDim ? a.dim : D, vdim = kAnyDim ? a.vdim : D;

    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid / kWave);
    // wave w takes query group w % QW and key tile kpart of every step
    const uint32_t qgroup = wave % QW, kpart = wave / QW;
    const uint32_t col = lane & 31, half = lane >> 5;
    // the lane's transpose-read address in a V tile (chunk 0, d tile 0)
    const uint32_t v_lane =
        (4 * (lane / 32) + (lane % 16) / 4) * VROW + 16 * ((lane / 16) % 2) + 4 * (lane % 4);
    const FlashItem item = flash_item(a, blockIdx.x);
    const uint32_t qblock = item.qblock, bh = item.bh;
    const uint32_t head = bh % a.qh, b = bh / a.qh;
    const size_t kv_base = ((size_t)b * a.kvh + head / a.group) * a.kl;
    const uint32_t qw = qblock * BM + qgroup * 32;      // the wave's first query
    const uint32_t qi = qw + col;                       // the lane's query
    const bool q_live = qi < a.ql;
    const float neg_inf = -__builtin_inff();

    half8 qf[KC];
    {
        const _Float16 *qrow = q + ((size_t)bh * a.ql + (q_live ? qi : 0)) * dim;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            const bool in_row = !kAnyDim || 16 * c + 8 * half < dim;
            qf[c] = *reinterpret_cast<const half8 *>(qrow + (in_row ? 16 * c + 8 * half : 0));
            if (!in_row) qf[c] = half8{};
        }
    }
    // wait for Q here: otherwise the wait analysis of the tile loop cannot
    // tell these loads from the next tile's prefetch and makes every S^T MFMA
    // wait for one more of the prefetch loads
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
    __builtin_amdgcn_sched_barrier(0);
    float16v o[VT];
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] = 0.0f;
    float m = neg_inf, l = 0.0f;   // running max (log2 units) and sum
    bool nan_seen = false;
    constexpr float kLog2e = 1.4426950408889634f;
    const float scale2 = a.scale * kLog2e;

    // key tiles any query of the block can see; this block's part of them
    const uint32_t all_tiles = flash_tiles(a.ql, a.kl, a.causal != 0, a.causal_offset, BM,
                                           kFlashN, qblock);
    const uint32_t share = (all_tiles + item.parts - 1) / item.parts;
    const uint32_t t_begin = min(item.part * share, all_tiles);
    const uint32_t tiles = min(t_begin + share, all_tiles);
    const bool wave_live = qw < a.ql;
    const uint64_t wave_last_key = (uint64_t)min(qw + 31, a.ql - 1) + a.causal_offset;
    const uint64_t lane_last_key = (uint64_t)qi + a.causal_offset;

    // tile loads of a step (KS tiles from key k0): thread `tid` moves vectors
    // tid, tid + THREADS, ... of K and of V (per tile row-major: key, 8-dim
    // group). The loads take no branch:
    // rows past the end are clamped onto the last key and zeroed when
    // stashed. (A fetch with a bounds-tested branch per load let the
    // compiler merge the whole-tile loads into that path, behind a wait for
    // every load just issued: the prefetch no longer overlapped the tile's
    // MFMAs, 15-20% slower.)
    half8 kreg[PER], vreg[PER];
    auto fetch = [&](uint32_t k0) {
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const uint32_t e = kWholeLoads ? tid + u * THREADS : min(tid + u * THREADS, VECS - 1u);
            const uint32_t tk = k0 + e / TV * kFlashN, r = e % TV;
            const size_t row = kv_base + min(tk + r / RV, a.kl - 1);
            const uint32_t c = r % RV * 8;
            // columns past the row are clamped onto its start (K's zeroed
            // when stashed; V's reach only output columns not stored)
            kreg[u] = *reinterpret_cast<const half8 *>(k + row * dim + (kAnyDim && c >= dim ? 0 : c));
            vreg[u] = *reinterpret_cast<const half8 *>(v + row * vdim + (kAnyDim && c >= vdim ? 0 : c));
        }
    };
    auto stash = [&](int buf, uint32_t k0) {
        if (k0 + KS * kFlashN > a.kl) {   // a ragged last step: zero the rows past the end
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                const uint32_t e = tid + u * THREADS, tk = k0 + e / TV * kFlashN, r = e % TV;
                if (tk + r / RV >= a.kl) {
                    kreg[u] = half8{};
                    vreg[u] = half8{};
                }
            }
        }
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const uint32_t e = tid + u * THREADS, tile = e / TV, r = e % TV;
            if (!kWholeLoads && e >= VECS) continue;
            if (kAnyDim && r % RV * 8 >= dim) kreg[u] = half8{};
            *reinterpret_cast<half8 *>(&ks[buf][tile * KTILE + (r / RV) * KROW + (r % RV) * 8]) = kreg[u];
            *reinterpret_cast<half8 *>(&vs[buf][tile * VTILE + (r / RV) * VROW + (r % RV) * 8]) = vreg[u];
        }
    };

    if (t_begin < tiles) {
        fetch(t_begin * kFlashN);
        stash(0, t_begin * kFlashN);
    }
    __syncthreads();
    // step: KS tiles from t0; this wave takes tile t0 + kpart
    for (uint32_t t0 = t_begin, step = 0; t0 < tiles; t0 += KS, ++step) {
        const int buf = step & 1;
        const uint32_t t = t0 + kpart;
        const uint32_t k0 = t * kFlashN;
        const bool more = t0 + KS < tiles;
        // The mask of the wave's scores: a lane pair's 16 keys of a row are two
        // 16-byte vectors (at any 2-byte alignment), whose middle quads change
        // lanes afterwards. Asked for before the next step's tiles, so that the
        // wait for them leaves those in flight (and no branch lies between).
        // A 2-byte load per score, each behind its own bounds test, bound the
        // masked kernels (us, before -> now: 32q/8kv 2048 x 2048 D 128 308 -> 101,
        // D 64 284 -> 77; with the second key part that the freed registers
        // allow, 12 heads 1024 x 1024 D 64 77 -> 16, unmasked 14).
        u32x4 mvec[kMask ? 4 : 1];
        if constexpr (kMask) {
            const _Float16 *mrow = mask + (size_t)(q_live ? qi : 0) * a.kl;
            if (mask != nullptr && k0 + kFlashN <= a.kl) {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    mvec[j] = *reinterpret_cast<const u32x4_2 *>(mrow + k0 + 16 * j + 8 * half);
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    mvec[j] = u32x4{0, 0, 0, 0};
                    if (mask == nullptr) continue;
                    half8 e;   // keys past the end read the last one
#pragma unroll
                    for (int i = 0; i < 8; ++i) e[i] = mrow[min(k0 + 16 * j + 8 * half + i, a.kl - 1)];
                    mvec[j] = __builtin_bit_cast(u32x4, e);
                }
            }
        }
        if (kMask || more) fetch((t0 + KS) * kFlashN);
        if (t < tiles && wave_live && !(a.causal && (uint64_t)k0 > wave_last_key)) {
            // interior tile: every key exists and is visible to every query of
            // the wave, so no per-score bounds or causal test is needed
            const bool interior = k0 + kFlashN <= a.kl &&
                                  (!a.causal || (uint64_t)k0 + kFlashN - 1 <= (uint64_t)qw + a.causal_offset);
            // the two 32-key halves are independent accumulation chains:
            // interleaved, each MFMA's latency is covered by the other's
            float16v st[2];
#pragma unroll
            for (int hblk = 0; hblk < 2; ++hblk)
#pragma unroll
                for (int r = 0; r < 16; ++r) st[hblk][r] = 0.0f;
            mfma_phase_begin();
#pragma unroll
            for (int c = 0; c < KC; ++c)
#pragma unroll
                for (int hblk = 0; hblk < 2; ++hblk) {
                    const half8 kf = *reinterpret_cast<const half8 *>(
                        &ks[buf][kpart * KTILE + (32 * hblk + col) * KROW + 16 * c + 8 * half]);
                    st[hblk] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[c], st[hblk], 0, 0, 0);
                }
            lds_read_ahead<2 * KC>();
            mfma_phase_end();
            // Scores are in log2 units: s = raw * scale2 (+ mask * log2 e).
            // Without a mask (and with scale2 > 0) st keeps the raw products
            // and sc = scale2 is applied inside exp2's fma; max_r(raw) * scale2
            // == max_r(raw * scale2) since rounding is monotone. The kMask
            // variant (also run for a scale <= 0, with or without a mask)
            // turns st into s and uses sc = 1 (fma(s, 1, -m) == s - m). The
            // interior test is taken once per tile (inside the unrolled loop
            // it became one branch per score).
            // kAnyDim keeps s in natural units and takes log2 e into sc: a mask
            // of the type's lowest value leaves scores near -65504 with steps of
            // 2^-8, the same in log2 units (-94502) with steps of 2^-7 (rows of
            // such scores alone: relative error 1.57e-3, in natural units 1.14e-3).
            auto score = [&](float raw, float add, uint32_t kk, bool edge) {
                float s = kAnyDim ? raw * a.scale + add : __builtin_fmaf(add, kLog2e, raw * scale2);
                if (edge && (kk >= a.kl || (a.causal && (uint64_t)kk > lane_last_key)))
                    s = neg_inf;
                return s;
            };
            // the online-softmax step for scores sv (s = sv * sc): P of the
            // tile into pf, m, l and o updated
            // (kAnyDim: P keeps f32 accuracy as an f16 pair, pf + pl)
            half8 pf[4], pl[kAnyDim ? 4 : 1];
            auto softmax = [&](const float16v (&sv)[2], float sc) {
                // four independent max chains instead of one of 32
                float part_max[4] = {neg_inf, neg_inf, neg_inf, neg_inf};
#pragma unroll
                for (int r = 0; r < 32; ++r) part_max[r % 4] = fmaxf(part_max[r % 4], sv[r / 16][r % 16]);
                const float tile_max =
                    pair_max(fmaxf(fmaxf(part_max[0], part_max[1]), fmaxf(part_max[2], part_max[3]))) * sc;
                // Lazy rescale: the running max m (and with it o and l) moves
                // only when some lane's maximum grows by more than
                // 2^kLazyLog2; until then p = 2^(s - m) <= 2^kLazyLog2, well
                // inside f16's range.
                const float m_cand = fmaxf(m, tile_max);
                if (__builtin_amdgcn_ballot_w64(m_cand > m + kLazyLog2) != 0) {
                    const float alpha = m_cand == neg_inf ? 1.0f : __builtin_amdgcn_exp2f(m - m_cand);
                    l *= alpha;
#pragma unroll
                    for (int tt = 0; tt < VT; ++tt)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o[tt][r] *= alpha;
                    m = m_cand;
                }
                const bool none = m == neg_inf;   // nothing visible to this query yet
                if (wave_any(none)) {
                    // a NaN score while nothing is visible is remembered: the
                    // row is NaN if a key becomes visible later (its p, NaN,
                    // also reaches o and l)
                    bool local_nan = false;
#pragma unroll
                    for (int r = 0; r < 32; ++r) local_nan = local_nan || sv[r / 16][r % 16] != sv[r / 16][r % 16];
                    nan_seen = nan_seen || (none && local_nan);
                }
                // with nothing visible every non-NaN score is -inf: p = 2^-inf = 0
                const float m_use = none ? 0.0f : m;
                if constexpr (kAnyDim) {
                    float part_sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int r = 0; r < 32; ++r) {
                        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[r / 16][r % 16], sc, -m_use));
                        part_sum[r % 4] += p;
                        pf[r / 8][r % 8] = (_Float16)p;
                        pl[r / 8][r % 8] = (_Float16)(p - (float)pf[r / 8][r % 8]);
                    }
                    l += pair_sum((part_sum[0] + part_sum[1]) + (part_sum[2] + part_sum[3]));
                    return;
                }
#pragma unroll
                for (int r = 0; r < 32; ++r)
                    pf[r / 8][r % 8] = (_Float16)__builtin_amdgcn_exp2f(__builtin_fmaf(sv[r / 16][r % 16], sc, -m_use));
                // the row sum of P as the MFMA sees it (f16), by v_dot2 with {1, 1}
                const half2_t ones = {(_Float16)1.0f, (_Float16)1.0f};
                float part_sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        part_sum[j] = __builtin_amdgcn_fdot2(half2_t{pf[c][2 * j], pf[c][2 * j + 1]}, ones,
                                                             part_sum[j], false);
                l += pair_sum((part_sum[0] + part_sum[1]) + (part_sum[2] + part_sum[3]));
            };
            if constexpr (kMask) {
                float16v sv[2];
                // quad of scores g of half-tile hblk: keys 32 hblk + 8 g + 4 half ..
                half4 mq[2][4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const auto x = __builtin_amdgcn_permlane32_swap(mvec[j].x, mvec[j].z, false, false);
                    const auto y = __builtin_amdgcn_permlane32_swap(mvec[j].y, mvec[j].w, false, false);
                    const unsigned x0 = x[0], x1 = x[1], y0 = y[0], y1 = y[1];
                    mq[j / 2][2 * (j % 2)] = __builtin_bit_cast(half4, uint2{x0, y0});
                    mq[j / 2][2 * (j % 2) + 1] = __builtin_bit_cast(half4, uint2{x1, y1});
                }
                if (interior) {
#pragma unroll
                    for (int hblk = 0; hblk < 2; ++hblk)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            sv[hblk][r] = score(st[hblk][r], (float)mq[hblk][r / 4][r % 4],
                                                k0 + 32 * hblk + 8 * (r / 4) + 4 * half + r % 4, false);
                } else {
#pragma unroll
                    for (int hblk = 0; hblk < 2; ++hblk)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            sv[hblk][r] = score(st[hblk][r], (float)mq[hblk][r / 4][r % 4],
                                                k0 + 32 * hblk + 8 * (r / 4) + 4 * half + r % 4, true);
                }
                softmax(sv, kAnyDim ? kLog2e : 1.0f);
            } else {
                // raw products, scale2 > 0: keys out of range or past the
                // causal limit become -inf in place
                if (!interior) {
#pragma unroll
                    for (int hblk = 0; hblk < 2; ++hblk)
#pragma unroll
                        for (int r = 0; r < 16; ++r) {
                            const uint32_t kk = k0 + 32 * hblk + 8 * (r / 4) + 4 * half + r % 4;
                            if (kk >= a.kl || (a.causal && (uint64_t)kk > lane_last_key)) st[hblk][r] = neg_inf;
                        }
                }
                softmax(st, scale2);
            }
            // the VT output tiles are independent chains: issue them side by side
            mfma_phase_begin();
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int tt = 0; tt < VT; ++tt) {
                    const _Float16 *vp = &vs[buf][kpart * VTILE + 16 * c * VROW + v_lane + 32 * tt];
                    const half4 lo = lds_read_tr(vp), hi = lds_read_tr(vp + 8 * VROW);
                    const half8 vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                    o[tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf[c], o[tt], 0, 0, 0);
                    if constexpr (kAnyDim)
                        o[tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pl[c], o[tt], 0, 0, 0);
                }
            lds_read_ahead<4 * VT, 2, kAnyDim ? 2 : 1>();
            mfma_phase_end();
        }
        if (more) stash(buf ^ 1, (t0 + KS) * kFlashN);
        __syncthreads();
    }
    // (the exchange outside the ||: short-circuited, lanes holding a NaN would
    // be inactive and send nothing)
    const int partner_nan = __shfl_xor((int)nan_seen, 32, kWave);
    nan_seen = nan_seen || partner_nan != 0;
    if constexpr (KS == 2) {
        // Merge the two key parts of each query group through LDS (the loop
        // ended on a barrier, so the tile buffers are free): the part-1 wave
        // leaves its (o, m, l, NaN flag), the part-0 wave folds them in with
        // the merge rules of sdpa_combine_kernel and goes on alone.
        static_assert(QW * (VT * 4 + 1) * kWave * 16 <= sizeof(tiles_lds), "merge area");
        f32x4 *xch = reinterpret_cast<f32x4 *>(tiles_lds) + qgroup * (VT * 4 + 1) * kWave + lane;
        if (kpart == 1) {
#pragma unroll
            for (int tt = 0; tt < VT; ++tt)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    xch[(tt * 4 + g) * kWave] =
                        f32x4{o[tt][4 * g], o[tt][4 * g + 1], o[tt][4 * g + 2], o[tt][4 * g + 3]};
            xch[VT * 4 * kWave] = f32x4{m, l, nan_seen ? 1.0f : 0.0f, 0.0f};
        }
        __syncthreads();
        if (kpart == 1) return;
        const f32x4 other = xch[VT * 4 * kWave];
        const float big = fmaxf(m, other.x);
        // weights 2^(m_s - M); a part that saw nothing (m_s = -inf), and
        // every part of a row whose M is not finite (a zero row), weigh 0
        const bool finite = __builtin_isfinite(big);
        const float w0 = !finite || m == -__builtin_inff() ? 0.0f : __builtin_amdgcn_exp2f(m - big);
        const float w1 = !finite || other.x == -__builtin_inff() ? 0.0f
                                                                  : __builtin_amdgcn_exp2f(other.x - big);
#pragma unroll
        for (int tt = 0; tt < VT; ++tt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 p = xch[(tt * 4 + g) * kWave];
#pragma unroll
                for (int j = 0; j < 4; ++j) o[tt][4 * g + j] = w0 * o[tt][4 * g + j] + w1 * p[j];
            }
        l = w0 * l + w1 * other.y;
        m = big;
        nan_seen = nan_seen || other.z != 0.0f;
    }
    if (!kAnyDim && !q_live) return;
    if constexpr (kSplit) {
        if (item.parts > 1) {
            if (q_live)
                write_partial<VT, kAnyDim>(a, item.part, (size_t)bh * a.ql + qi, half, o, m, l, nan_seen);
            return;
        }
    }
    const bool zero = !__builtin_isfinite(m);
    const float inverse = l == 0.0f ? 0.0f : 1.0f / l;
    const float nan = __builtin_nanf("");
    _Float16 *orow = out + ((size_t)bh * a.ql + qi) * vdim;
    float finite = 0.0f;   // 0 * x is NaN for a non-finite x
#pragma unroll
    for (int tt = 0; tt < VT; ++tt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (kAnyDim && (!q_live || 32 * tt + 8 * g + 4 * half >= vdim)) continue;
            _Float16 quad[4] __attribute__((aligned(8)));
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (kAnyDim) finite = __builtin_fmaf(0.0f, o[tt][4 * g + j], finite);
                quad[j] = (_Float16)(zero ? 0.0f : nan_seen ? nan : o[tt][4 * g + j] * inverse);
            }
            *reinterpret_cast<uint2 *>(orow + 32 * tt + 8 * g + 4 * half) =
                *reinterpret_cast<const uint2 *>(quad);
        }
    if constexpr (kAnyDim) {
        // An infinite V element meets the halves of P as hi + lo, of which lo
        // may be negative or zero and hi rounded to zero where P is positive:
        // inf - inf or 0 * inf. A row with a finite sum and an output that is
        // not finite is done again by the row routine.
        uint64_t redo = __builtin_amdgcn_ballot_w64(q_live && !zero && !nan_seen && finite != 0.0f &&
                                                    __builtin_isfinite(l));
        redo = (redo | redo >> 32) & 0xffffffffu;
        if (redo != 0) __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);   // the stores above come first
#pragma unroll 1
        while (redo != 0) {
            const uint32_t c = (uint32_t)__builtin_ctzll(redo);
            redo &= redo - 1;
            sdpa_row<_Float16, true>(q, k, v, mask, out, a, (size_t)bh * a.ql + qw + c, lane);
        }
    }
}

// f32 flash kernel (D = Dv in {64, 128}): v_mfma_f32_32x32x2_f32, one wave
// per 32 queries, BM queries per block, 32-key K and V tiles in LDS
// (row-major, row pitch D + 4 floats: conflict-free 16-byte reads),
// double-buffered.
//   S^T = K Q^T: MFMA c contracts the d pair {c, D/2 + c}: lane half h holds
//   d in [h D/2, (h + 1) D/2), so each lane's K and Q operands are runs of
//   consecutive floats (Q stays in registers for the whole kernel).
//   out^T += V^T P^T: MFMA j contracts the key pair {8(j/4) + j%4, that + 4},
//   exactly the keys that accumulator register j of S^T holds in the two lane
//   halves, so P is the B operand as it stands and V needs no transpose.
// Scores are s * scale (+ mask), causal keys -inf; the online softmax uses
// expf (libm accuracy) and normalises once at the end by the reciprocal of
// the sum, with the special-row rules of the f16 kernel.
constexpr int kFlashN32 = 32;   // keys per f32 tile

template <int D, int BM, bool kMask, bool kSplit, int KS, bool kAnyDim = false>
__global__ __launch_bounds__(BM * 2 * KS) void sdpa_flash_f32_kernel(const float *__restrict__ q,
                                                                const float *__restrict__ k,
                                                                const float *__restrict__ v,
                                                                const float *__restrict__ mask,
                                                                float *__restrict__ out,
                                                                SdpaArgs a) {
    constexpr int QW = BM / 32;              // query groups of 32: one wave each per key part
    constexpr int THREADS = BM * 2 * KS;
    constexpr int KN = kFlashN32;
    constexpr int VT = (D + 31) / 32;        // 32-row tiles of out^T
    constexpr int ROW = 32 * VT + 4;         // LDS row (floats)
    constexpr int QC = D / 2;                // MFMAs of S^T per tile
    constexpr int TILE = KN * ROW;           // LDS floats of one K or V tile
    constexpr int TV = KN * D / 4;           // float4 vectors per K or V tile
    constexpr int VECS = KS * TV;            // per operand and step (KS tiles)
    constexpr int PER = (VECS + THREADS - 1) / THREADS;
    constexpr bool kWholeLoads = VECS % THREADS == 0;
    static_assert(kWholeLoads || kAnyDim, "tile load split");
    constexpr int RV = D / 4;                // float4 vectors per LDS row
    const uint32_t dim = kAnyDim ? a.dim : D, vdim = kAnyDim ? a.vdim : D;
    // step buffer b: K tiles at lds[b * 2 KS TILE], V tiles KS TILE further
    __shared__ __attribute__((aligned(16))) float lds[2 * 2 * KS * TILE];

    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(tid / kWave);
    // wave w takes query group w % QW and key tile kpart of every step
    const uint32_t qgroup = wave % QW, kpart = wave / QW;
    const uint32_t col = lane & 31, half = lane >> 5;
    const FlashItem item = flash_item(a, blockIdx.x);
    const uint32_t qblock = item.qblock, bh = item.bh;
    const uint32_t head = bh % a.qh, b = bh / a.qh;
    const size_t kv_base = ((size_t)b * a.kvh + head / a.group) * a.kl;
    const uint32_t qw = qblock * BM + qgroup * 32;
    const uint32_t qi = qw + col;
    const bool q_live = qi < a.ql;
    const float neg_inf = -__builtin_inff();

    float qf[QC];
    {
        const f32x4 *qrow = reinterpret_cast<const f32x4 *>(
            q + ((size_t)bh * a.ql + (q_live ? qi : 0)) * dim);
#pragma unroll
        for (int c = 0; c < QC / 4; ++c) {
            const uint32_t at = half * (QC / 4) + c;
            const bool in_row = !kAnyDim || 4 * at < dim;
            f32x4 t = qrow[in_row ? at : 0];
            if (!in_row) t = f32x4{0, 0, 0, 0};
            qf[4 * c] = t.x;
            qf[4 * c + 1] = t.y;
            qf[4 * c + 2] = t.z;
            qf[4 * c + 3] = t.w;
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);   // Q ready before the tile loop
    __builtin_amdgcn_sched_barrier(0);
    float16v o[VT];
#pragma unroll
    for (int t = 0; t < VT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[t][r] = 0.0f;
    float m = neg_inf, l = 0.0f;
    bool nan_seen = false;

    const uint32_t all_tiles = flash_tiles(a.ql, a.kl, a.causal != 0, a.causal_offset, BM, KN,
                                           qblock);
    const uint32_t share = (all_tiles + item.parts - 1) / item.parts;
    const uint32_t t_begin = min(item.part * share, all_tiles);
    const uint32_t tiles = min(t_begin + share, all_tiles);
    const bool wave_live = qw < a.ql;
    const uint64_t wave_last_key = (uint64_t)min(qw + 31, a.ql - 1) + a.causal_offset;
    const uint64_t lane_last_key = (uint64_t)qi + a.causal_offset;

    // tile loads of a step (KS tiles from key k0): vector e of a tile is key
    // e / (D/4), floats 4 (e % (D/4)) ...; branch-free (rows past the end
    // clamped onto the last key, zeroed when stored: see the f16 kernel)
    f32x4 kreg[PER], vreg[PER];
    auto fetch = [&](uint32_t k0) {
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const uint32_t e = kWholeLoads ? tid + u * THREADS : min(tid + u * THREADS, VECS - 1u);
            const uint32_t tk = k0 + e / TV * KN, r = e % TV;
            const size_t row = kv_base + min(tk + r / RV, a.kl - 1);
            const uint32_t c = r % RV * 4;
            kreg[u] = *reinterpret_cast<const f32x4 *>(k + row * dim + (kAnyDim && c >= dim ? 0 : c));
            vreg[u] = *reinterpret_cast<const f32x4 *>(v + row * vdim + (kAnyDim && c >= vdim ? 0 : c));
        }
    };
    auto stash = [&](int buf, uint32_t k0) {
        if (k0 + KS * KN > a.kl) {   // a ragged last step: zero the rows past the end
#pragma unroll
            for (int u = 0; u < PER; ++u) {
                const uint32_t e = tid + u * THREADS, tk = k0 + e / TV * KN, r = e % TV;
                if (tk + r / RV >= a.kl) {
                    kreg[u] = f32x4{0, 0, 0, 0};
                    vreg[u] = f32x4{0, 0, 0, 0};
                }
            }
        }
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const uint32_t e = tid + u * THREADS, r = e % TV;
            if (!kWholeLoads && e >= VECS) continue;
            if (kAnyDim && r % RV * 4 >= dim) kreg[u] = f32x4{0, 0, 0, 0};
            const uint32_t at = buf * 2 * KS * TILE + (e / TV) * TILE + (r / RV) * ROW + (r % RV) * 4;
            *reinterpret_cast<f32x4 *>(&lds[at]) = kreg[u];
            *reinterpret_cast<f32x4 *>(&lds[at + KS * TILE]) = vreg[u];
        }
    };

    if (t_begin < tiles) {
        fetch(t_begin * KN);
        stash(0, t_begin * KN);
    }
    __syncthreads();
    // step: KS tiles from t0; this wave takes tile t0 + kpart
    for (uint32_t t0 = t_begin, step = 0; t0 < tiles; t0 += KS, ++step) {
        const int buf = step & 1;
        const uint32_t t = t0 + kpart;
        const uint32_t k0 = t * KN;
        const bool more = t0 + KS < tiles;
        // The mask of the wave's scores, asked for before the next step's tiles
        // (see the f16 kernel; 32q/8kv 2048 x 2048 D 64 500 -> 349 us). Unlike
        // there the last step has its branch: without it the D 128 form spilled 8
        // registers, and short key ranges fetched a tile more (us, without ->
        // with: 32q/8kv 2048 x 2048 670 -> 602, 8 x 32q/8kv 16 x 2048 323 -> 169, 512
        // x 4 heads 49 x 49 124 -> 95).
        f32x4 mq[kMask ? 4 : 1];
        if constexpr (kMask) {
            const float *mrow = mask + (size_t)(q_live ? qi : 0) * a.kl;
            if (!wave_live) {   // (dead waves of a last block only move tiles)
            } else if (k0 + KN <= a.kl) {
#pragma unroll
                for (int g = 0; g < 4; ++g) mq[g] = *reinterpret_cast<const f32x4_4 *>(mrow + k0 + 8 * g + 4 * half);
            } else {
#pragma unroll
                for (int g = 0; g < 4; ++g)
#pragma unroll
                    for (int i = 0; i < 4; ++i) mq[g][i] = mrow[min(k0 + 8 * g + 4 * half + i, a.kl - 1)];
            }
        }
        if (more) fetch((t0 + KS) * KN);
        const float *kt = &lds[buf * 2 * KS * TILE + kpart * TILE];   // this wave's K tile
        const float *vt = kt + KS * TILE;                              // and V tile
        if (t < tiles && wave_live && !(a.causal && (uint64_t)k0 > wave_last_key)) {
            const bool interior = k0 + KN <= a.kl &&
                                  (!a.causal || (uint64_t)k0 + KN - 1 <= (uint64_t)qw + a.causal_offset);
            // two accumulators (even and odd d pairs) keep two MFMA chains in flight
            float16v acc[2];
#pragma unroll
            for (int h2 = 0; h2 < 2; ++h2)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[h2][r] = 0.0f;
            const float *krow = kt + col * ROW + half * QC;
#pragma unroll
            for (int c4 = 0; c4 < QC / 4; ++c4) {
                const f32x4 kf = *reinterpret_cast<const f32x4 *>(krow + 4 * c4);
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.x, qf[4 * c4], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.y, qf[4 * c4 + 1], acc[1], 0, 0, 0);
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.z, qf[4 * c4 + 2], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf.w, qf[4 * c4 + 3], acc[1], 0, 0, 0);
            }
            float st[16];
            float local_max = neg_inf;
            auto score = [&](float raw, int r, uint32_t kk, bool edge) {
                float s = raw * a.scale;
                if constexpr (kMask) s = s + mq[r / 4][r % 4];
                if (edge && (kk >= a.kl || (a.causal && (uint64_t)kk > lane_last_key)))
                    s = neg_inf;
                return s;
            };
            float part_max[4] = {neg_inf, neg_inf, neg_inf, neg_inf};
            if (interior) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    st[r] = score(acc[0][r] + acc[1][r], r, k0 + 8 * (r / 4) + 4 * half + r % 4, false);
                    part_max[r % 4] = fmaxf(part_max[r % 4], st[r]);
                }
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    st[r] = score(acc[0][r] + acc[1][r], r, k0 + 8 * (r / 4) + 4 * half + r % 4, true);
                    part_max[r % 4] = fmaxf(part_max[r % 4], st[r]);
                }
            }
            local_max = fmaxf(fmaxf(part_max[0], part_max[1]), fmaxf(part_max[2], part_max[3]));
            const float m_new = fmaxf(m, pair_max(local_max));
            const bool none = m_new == neg_inf;
            if (wave_any(none)) {
                bool local_nan = false;
#pragma unroll
                for (int r = 0; r < 16; ++r) local_nan = local_nan || st[r] != st[r];
                nan_seen = nan_seen || (none && local_nan);
            }
            const float alpha = none ? 1.0f : expf(m - m_new);
            float part_sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                st[r] = none ? 0.0f : expf(st[r] - m_new);
                part_sum[r % 4] += st[r];
            }
            const float local_sum = (part_sum[0] + part_sum[1]) + (part_sum[2] + part_sum[3]);
            l = l * alpha + pair_sum(local_sum);
            m = m_new;
            if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
                for (int tt = 0; tt < VT; ++tt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[tt][r] *= alpha;
            }
            // the VT output tiles are independent chains: issue them side by side
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const float *vrow = vt + (8 * (j / 4) + 4 * half + j % 4) * ROW + col;
#pragma unroll
                for (int tt = 0; tt < VT; ++tt)
                    o[tt] = __builtin_amdgcn_mfma_f32_32x32x2f32(vrow[32 * tt], st[j], o[tt], 0, 0, 0);
            }
        }
        if (more) stash(buf ^ 1, (t0 + KS) * KN);
        __syncthreads();
    }
    // (the exchange outside the ||: short-circuited, lanes holding a NaN would
    // be inactive and send nothing)
    const int partner_nan = __shfl_xor((int)nan_seen, 32, kWave);
    nan_seen = nan_seen || partner_nan != 0;
    if constexpr (KS == 2) {
        // the two key parts of each query group merged through LDS, as in
        // the f16 kernel, with natural-exp weights e^(m_s - M)
        static_assert(QW * (VT * 4 + 1) * kWave * 16 <= sizeof(lds), "merge area");
        f32x4 *xch = reinterpret_cast<f32x4 *>(&lds[0]) + qgroup * (VT * 4 + 1) * kWave + lane;
        if (kpart == 1) {
#pragma unroll
            for (int tt = 0; tt < VT; ++tt)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    xch[(tt * 4 + g) * kWave] =
                        f32x4{o[tt][4 * g], o[tt][4 * g + 1], o[tt][4 * g + 2], o[tt][4 * g + 3]};
            xch[VT * 4 * kWave] = f32x4{m, l, nan_seen ? 1.0f : 0.0f, 0.0f};
        }
        __syncthreads();
        if (kpart == 1) return;
        const f32x4 other = xch[VT * 4 * kWave];
        const float big = fmaxf(m, other.x);
        const bool finite = __builtin_isfinite(big);
        const float w0 = !finite || m == -__builtin_inff() ? 0.0f : expf(m - big);
        const float w1 = !finite || other.x == -__builtin_inff() ? 0.0f : expf(other.x - big);
#pragma unroll
        for (int tt = 0; tt < VT; ++tt)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 p = xch[(tt * 4 + g) * kWave];
#pragma unroll
                for (int j = 0; j < 4; ++j) o[tt][4 * g + j] = w0 * o[tt][4 * g + j] + w1 * p[j];
            }
        l = w0 * l + w1 * other.y;
        m = big;
        nan_seen = nan_seen || other.z != 0.0f;
    }
    if (!q_live) return;
    if constexpr (kSplit) {
        if (item.parts > 1) {
            write_partial<VT, kAnyDim>(a, item.part, (size_t)bh * a.ql + qi, half, o, m, l, nan_seen);
            return;
        }
    }
    const bool zero = !__builtin_isfinite(m);
    const float inverse = l == 0.0f ? 0.0f : 1.0f / l;
    const float nan = __builtin_nanf("");
    float *orow = out + ((size_t)bh * a.ql + qi) * vdim;
#pragma unroll
    for (int tt = 0; tt < VT; ++tt)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (kAnyDim && 32 * tt + 8 * g + 4 * half >= vdim) continue;
            f32x4 quad;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                quad[j] = zero ? 0.0f : nan_seen ? nan : o[tt][4 * g + j] * inverse;
            *reinterpret_cast<f32x4 *>(orow + 32 * tt + 8 * g + 4 * half) = quad;
        }
}

// Head dims other than 64 and 128 (k_attention_dims.hip): one launch of the
// kernel compiled for `variant`; the caller sizes the grid and the block.
struct FlashVariant {
    uint32_t dim, bm, key_parts;
    bool general, split;
};
hipError_t launch_any_dim_f16(const FlashVariant &variant, dim3 grid, dim3 block, hipStream_t s,
                              const _Float16 *q, const _Float16 *k, const _Float16 *v,
                              const _Float16 *mask, _Float16 *out, const SdpaArgs &a);
hipError_t launch_any_dim_f32(const FlashVariant &variant, dim3 grid, dim3 block, hipStream_t s,
                              const float *q, const float *k, const float *v, const float *mask,
                              float *out, const SdpaArgs &a);

}  // namespace flash
}  // namespace icsdk
