// Attention of few query rows against a long key range (decoding, short
// chunks): the query heads of one kv head are packed into one tile of rows, so
// K and V are read once per kv head, and the key range is spread over waves
// and blocks.
//
// The rows of a kv head -- its `group` query heads times q_len positions -- are
// consecutive in q and out, so packed row r is row r of a [group * q_len, D]
// matrix; its position is r % q_len. A wave holds 16 rows (more rows: more
// blocks, which read K and V from the caches; 32 or 64 rows per wave measured
// slower, one wave per SIMD) and walks key tiles of 32 (f16) or 16 (f32) keys;
// a block's four waves take every fourth tile of the block's part of the keys,
// with nothing shared until the end: K and V go from memory straight into the
// MFMA operands' registers, the next tile's loads issued before the current
// tile is computed. No LDS, no barrier in the loop.
//
// v_mfma_f32_16x16x32_f16 (f16) and 16x16x4_f32: A[m][k] in lane l at m = l %
// 16, k = 8 g + i (f32: k = g), g = l / 16; B[k][n] at n = l % 16 likewise;
// D[m][n] at n = l % 16, m = 4 g + r.
//   Scores S^T = K Q^T: A row m of sub-tile s is key 4 NS (m / 4) + 4 s + m %
//   4 of the tile (NS sub-tiles of 16 keys), so lane l holds, of row l % 16,
//   the keys 4 NS g .. 4 NS g + 4 NS - 1: consecutive, and exactly the keys
//   that its lane group supplies in the next product.
//   out^T = V^T P^T: the contraction runs over those keys, so P is the B
//   operand as it stands. The lane loads vector m = l % 16 (VE elements) of
//   the V rows of its group's keys; MFMA j takes element j of them, so
//   out^T row m of MFMA j is column VE m + j (f16: the 8 keys' elements j
//   are gathered by v_perm, one per two; f32: each MFMA takes one key per
//   group). Columns past the head dim load column 0 again and are not stored.
// Softmax as in the flash kernel: log2 units (f32, masked f16: natural), lazy rescale, NaN
// flag for rows that have seen nothing yet; f16 P is the pair hi + lo. Each
// lane sums its own keys; lane groups meet at the end. Waves merge through
// LDS, parts through sdpa_fold_kernel. A row with a finite sum and an output
// that is not finite (an infinite value; keys past the end read the last row
// again) is done again by the row routine.
//
// Bound: HBM bytes of K and V, or for short ranges the launches and one
// wave's chain. Measured (us, flash kernel with a block per query head ->
// here): f16 D 128 8 x 32q/8kv over 4096 keys 79 -> 26 (5.2 TB/s), 32 x 32q/8kv
// over 2048 160 -> 41 (6.5 TB/s), 32q/8kv over 16384 37 -> 17, over 2048 11.4 ->
// 9.6; f32 D 128 8 x 32q/8kv over 4096 314 -> 48.
#include "flash.hpp"
#include "decode.hpp"

#include <type_traits>

namespace icsdk {
namespace flash {
namespace {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kDecodeWaves = 4;
constexpr float kLog2e = 1.4426950408889634f;

template <typename S> constexpr int sub_tiles() { return sizeof(S) == 2 ? 2 : 1; }

// Max / sum over the four lanes (one per group) that hold one row.
__device__ inline float groups_max(float v) {
    v = fmaxf(v, __shfl_xor(v, 16, kWave));
    return fmaxf(v, __shfl_xor(v, 32, kWave));
}
__device__ inline float groups_sum(float v) {
    v += __shfl_xor(v, 16, kWave);
    return v + __shfl_xor(v, 32, kWave);
}

// One key tile of K and V in registers. KC: 32-dim (f16) or 16-dim (f32)
// chunks of a K row; V rows are VC chunks of 16 vectors of VE elements.
template <typename S, int KC, int VE, int VC> struct KvTile {
    static constexpr int NS = sub_tiles<S>();
    static constexpr int KEYS = 4 * NS;               // keys per lane
    static constexpr int E = 16 / sizeof(S);
    using VVec = std::conditional_t<VE * sizeof(S) == 16, u32x4, u32x2>;
    u32x4 k[NS][KC];
    VVec v[VC][KEYS];

    // rows past the last key read the last one, columns past the head dim
    // column 0 (zeroed by pad())
    __device__ inline void load(const S *kbase, const S *vbase, uint32_t key0, uint32_t kl,
                                uint32_t dim, uint32_t vdim, uint32_t g, uint32_t m) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const uint32_t key = min(key0 + 4 * NS * (m / 4) + 4 * s + m % 4, kl - 1);
            const S *row = kbase + (size_t)key * dim;
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                const uint32_t d = 4 * E * c + E * g;
                k[s][c] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(row + (d < dim ? d : 0)));
            }
        }
#pragma unroll
        for (int i = 0; i < KEYS; ++i) {
            const uint32_t key = min(key0 + KEYS * g + i, kl - 1);
            const S *row = vbase + (size_t)key * vdim;
#pragma unroll
            for (int t = 0; t < VC; ++t) {
                const uint32_t d = 16 * VE * t + VE * m;
                v[t][i] = __builtin_nontemporal_load(reinterpret_cast<const VVec *>(row + (d < vdim ? d : 0)));
            }
        }
    }
    __device__ inline void pad(uint32_t dim, uint32_t g) {
#pragma unroll
        for (int c = 0; c < KC; ++c)
            if (4 * E * c + E * g >= dim)
#pragma unroll
                for (int s = 0; s < NS; ++s) k[s][c] = u32x4{0, 0, 0, 0};
    }
};

template <typename S, int KC, int VE, int VC, bool kMask>
__global__ __launch_bounds__(kDecodeWaves *kWave) void sdpa_decode_kernel(
    const S *__restrict__ q, const S *__restrict__ k, const S *__restrict__ v,
    const S *__restrict__ mask, S *__restrict__ out, SdpaArgs a, DecodeArgs da) {
    constexpr bool kHalf = sizeof(S) == 2;
    using Tile = KvTile<S, KC, VE, VC>;
    constexpr int NS = Tile::NS, KEYS = Tile::KEYS, E = Tile::E, NJ = VE * VC;
    constexpr uint32_t kTileKeys = 16 * NS;
    __shared__ f32x4 lds_o[kDecodeWaves][NJ][kWave];
    __shared__ f32x4 lds_ml[kDecodeWaves][16];
    const uint32_t lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    // block -> (batch * kvh + kv head, row group, part of the keys)
    const uint32_t part = blockIdx.x % da.parts, hr = blockIdx.x / da.parts;
    const uint32_t head = hr / da.row_groups, first_row = hr % da.row_groups * 16;
    const uint32_t rows = a.group * a.ql - first_row;   // from this group's first row on
    const size_t row0 = (size_t)head * (a.group * a.ql) + first_row;
    const S *kbase = k + (size_t)head * a.kl * a.dim;
    const S *vbase = v + (size_t)head * a.kl * a.vdim;
    const float neg_inf = -__builtin_inff();

    // keys any row sees, and this block's tiles of them
    const uint32_t seen = a.causal ? (uint32_t)min((uint64_t)a.ql + a.causal_offset, (uint64_t)a.kl) : a.kl;
    const uint32_t tiles = (seen + kTileKeys - 1) / kTileKeys;
    const uint32_t share = (tiles + da.parts - 1) / da.parts;
    const uint32_t t_begin = min(part * share, tiles), t_end = min(t_begin + share, tiles);

    Tile kv[2];
    uint32_t t = t_begin + wave;
    if (t < t_end) kv[0].load(kbase, vbase, t * kTileKeys, a.kl, a.dim, a.vdim, g, m);
    // Q operands; rows past the last one read it again (not stored)
    const uint32_t r = min(m, rows - 1), pos = (first_row + r) % a.ql;
    u32x4 qf[KC];
#pragma unroll
    for (int c = 0; c < KC; ++c) {
        const uint32_t d = 4 * E * c + E * g;
        qf[c] = *reinterpret_cast<const u32x4 *>(q + (row0 + r) * a.dim + (d < a.dim ? d : 0));
        if (d >= a.dim) qf[c] = u32x4{0, 0, 0, 0};
    }
    f32x4 o[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) o[j] = f32x4{0, 0, 0, 0};
    float mx = neg_inf, sum = 0.0f;
    bool nan_seen = false;
    // f16 scores are in log2 units, f32 and masked f16 scores in natural ones:
    // near a mask's -65504 those have the finer steps (2^-8; -94502 has 2^-7), and
    // `unit` then enters with the maximum's subtraction, in one fma. The maximum
    // is kept in the units of exp2 (f16) or expf (f32).
    constexpr float unit = kHalf && kMask ? kLog2e : 1.0f;
    const float scale = kHalf && !kMask ? a.scale * kLog2e : a.scale;

    auto power = [](float x) { return kHalf ? __builtin_amdgcn_exp2f(x) : expf(x); };
    // the last key the lane's row sees
    const uint32_t last_key =
        a.causal ? (uint32_t)min((uint64_t)pos + a.causal_offset, (uint64_t)a.kl - 1) : a.kl - 1;

    auto compute = [&](Tile &c, uint32_t key0) {
        if (a.dim != 4 * E * KC) c.pad(a.dim, g);
        const uint32_t first = key0 + KEYS * g;   // the lane's keys: first .. first + KEYS - 1
        float p[KEYS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            f32x4 acc = {0, 0, 0, 0};
#pragma unroll
            for (int ch = 0; ch < KC; ++ch) {
                if constexpr (kHalf) {
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, c.k[s][ch]),
                                                                 __builtin_bit_cast(half8, qf[ch]), acc, 0, 0, 0);
                } else {
                    const f32x4 kf = __builtin_bit_cast(f32x4, c.k[s][ch]), qv = __builtin_bit_cast(f32x4, qf[ch]);
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i], qv[i], acc, 0, 0, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) p[4 * s + i] = acc[i] * scale;
        }
        if constexpr (kMask) {
            const S *mrow = mask + (size_t)pos * a.kl;
            if (first + KEYS <= a.kl) {
                if constexpr (kHalf) {
                    const half8 mv = __builtin_bit_cast(half8, (u32x4)*reinterpret_cast<const u32x4_2 *>(mrow + first));
#pragma unroll
                    for (int i = 0; i < KEYS; ++i) p[i] = p[i] + (float)mv[i];
                } else {
                    const f32x4 mv = *reinterpret_cast<const f32x4_4 *>(mrow + first);
#pragma unroll
                    for (int i = 0; i < KEYS; ++i) p[i] = p[i] + mv[i];
                }
            } else {
#pragma unroll
                for (int i = 0; i < KEYS; ++i)
                    if (first + i < a.kl) p[i] = p[i] + (float)mrow[first + i];
            }
        }
        if (key0 + kTileKeys > a.kl || a.causal) {
#pragma unroll
            for (int i = 0; i < KEYS; ++i) p[i] = first + i > last_key ? neg_inf : p[i];
        }
        float big = neg_inf;
#pragma unroll
        for (int i = 0; i < KEYS; ++i) big = fmaxf(big, p[i]);
        big *= unit;
        // f16: the running maximum moves only when a row's grows by more than
        // 2^kLazyLog2 (p stays within f16)
        if (__builtin_amdgcn_ballot_w64(big > mx + (kHalf ? kLazyLog2 : 0.0f)) != 0) {
            const float now = groups_max(fmaxf(big, mx));
            const float alpha = now == neg_inf ? 1.0f : power(mx - now);
            sum *= alpha;
#pragma unroll
            for (int j = 0; j < NJ; ++j) o[j] *= alpha;
            mx = now;
        }
        const bool none = mx == neg_inf;
        if (wave_any(none)) {
            bool local_nan = false;
#pragma unroll
            for (int i = 0; i < KEYS; ++i) local_nan = local_nan || p[i] != p[i];
            nan_seen = nan_seen || (none && local_nan);
        }
        float add = 0.0f;
#pragma unroll
        for (int i = 0; i < KEYS; ++i) {
            p[i] = none ? 0.0f : power(kHalf && kMask ? __builtin_fmaf(p[i], unit, -mx) : p[i] - mx);
            add += p[i];
        }
        sum += add;
        if constexpr (kHalf) {
            half8 hi, lo;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                hi[i] = (_Float16)p[i];
                lo[i] = (_Float16)(p[i] - (float)hi[i]);
            }
#pragma unroll
            for (int tt = 0; tt < VC; ++tt)
#pragma unroll
                for (int j = 0; j < VE; ++j) {
                    u32x4 f;
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        f[i] = __builtin_amdgcn_perm(c.v[tt][2 * i + 1][j / 2], c.v[tt][2 * i][j / 2],
                                                     j % 2 ? 0x07060302u : 0x05040100u);
                    const half8 vf = __builtin_bit_cast(half8, f);
                    f32x4 &acc = o[tt * VE + j];
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, hi, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, lo, acc, 0, 0, 0);
                }
        } else {
#pragma unroll
            for (int i = 0; i < KEYS; ++i)
#pragma unroll
                for (int tt = 0; tt < VC; ++tt) {
                    const f32x4 vv = __builtin_bit_cast(f32x4, c.v[tt][i]);
#pragma unroll
                    for (int j = 0; j < VE; ++j)
                        o[tt * VE + j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vv[j], p[i], o[tt * VE + j], 0, 0, 0);
                }
        }
    };

    // two tiles per turn, each loaded while the one before is computed
    while (t < t_end) {
        const uint32_t t1 = t + kDecodeWaves, t2 = t1 + kDecodeWaves;
        if (t1 < t_end) kv[1].load(kbase, vbase, t1 * kTileKeys, a.kl, a.dim, a.vdim, g, m);
        compute(kv[0], t * kTileKeys);
        if (t1 >= t_end) break;
        if (t2 < t_end) kv[0].load(kbase, vbase, t2 * kTileKeys, a.kl, a.dim, a.vdim, g, m);
        compute(kv[1], t1 * kTileKeys);
        t = t2;
    }

    // merge the waves: every wave leaves its (max, sum, NaN flag) per row and
    // its outputs; wave w then folds register w of every output tile, columns
    // VE (4 g + w) .. + VE - 1 of each chunk
    sum = groups_sum(sum);
    const bool wave_nan = groups_max(nan_seen ? 1.0f : 0.0f) != 0.0f;
    if (g == 0) lds_ml[wave][m] = f32x4{mx, sum, wave_nan ? 1.0f : 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < NJ; ++j) lds_o[wave][j][lane] = o[j];
    __syncthreads();
    float w[kDecodeWaves], big = neg_inf, total = 0.0f;
    bool nan = false;
#pragma unroll
    for (int i = 0; i < kDecodeWaves; ++i) big = fmaxf(big, lds_ml[i][m].x);
    const bool finite = __builtin_isfinite(big);
#pragma unroll
    for (int i = 0; i < kDecodeWaves; ++i) {
        const f32x4 ml = lds_ml[i][m];
        w[i] = !finite || ml.x == neg_inf ? 0.0f : power(ml.x - big);
        total += w[i] * ml.y;
        nan = nan || ml.z != 0.0f;
    }
    const bool live = m < rows;
    const size_t row = row0 + r, all_rows = (size_t)a.batch * a.qh * a.ql;
    const float inverse = total == 0.0f ? 0.0f : 1.0f / total;
    float odd = 0.0f;   // 0 * x is NaN for a non-finite x
#pragma unroll
    for (int tt = 0; tt < VC; ++tt) {
        float val[VE];
        const uint32_t d = 16 * VE * tt + VE * (4 * g + wave);
        const bool in_row = d < a.vdim;
#pragma unroll
        for (int j = 0; j < VE; ++j) {
            val[j] = 0.0f;
#pragma unroll
            for (int i = 0; i < kDecodeWaves; ++i)
                val[j] += w[i] * reinterpret_cast<const float *>(&lds_o[i][tt * VE + j][lane])[wave];
            odd = in_row ? __builtin_fmaf(0.0f, val[j], odd) : odd;
        }
        if (!live || !in_row) continue;
        if (da.parts > 1) {
            float *prow = a.part_o + ((size_t)part * all_rows + row) * a.vdim + d;
#pragma unroll
            for (int j = 0; j < VE; j += 4)
                *reinterpret_cast<f32x4 *>(prow + j) = f32x4{val[j], val[j + 1], val[j + 2], val[j + 3]};
        } else {
            S res[VE] __attribute__((aligned(16)));
#pragma unroll
            for (int j = 0; j < VE; ++j)
                res[j] = (S)(!finite ? 0.0f : nan ? __builtin_nanf("") : val[j] * inverse);
            S *orow = out + row * a.vdim + d;
            if constexpr (VE * sizeof(S) == 16)
                *reinterpret_cast<u32x4 *>(orow) = *reinterpret_cast<const u32x4 *>(res);
            else
                *reinterpret_cast<u32x2 *>(orow) = *reinterpret_cast<const u32x2 *>(res);
        }
    }
    if (da.parts > 1) {
        if (wave == 0 && g == 0 && live)
            a.part_ml[(size_t)part * all_rows + row] = f32x4{big, total, nan ? 1.0f : 0.0f, 0.0f};
        return;
    }
    uint64_t redo = __builtin_amdgcn_ballot_w64(live && finite && !nan && odd != 0.0f && __builtin_isfinite(total));
    if (!__syncthreads_or(redo != 0)) return;   // (the stores above come first)
    redo |= redo >> 32;
    redo = (redo | redo >> 16) & 0xffffu;
#pragma unroll 1
    while (redo != 0) {
        const uint32_t c = (uint32_t)__builtin_ctzll(redo);
        redo &= redo - 1;
        sdpa_row<S, true>(q, k, v, mask, out, a, row0 + c, lane);
    }
}

// Folds the parts of a row, one block per row: thread (c, l) folds parts l, l +
// 256 / CG, ... of columns 4 c .. 4 c + 3, eight parts' loads in flight, and
// the part lanes meet in LDS. (One thread per four outputs walking all the
// parts took 16 of 28 us at 64 parts.) CG: a power of two >= vdim / 4.
template <typename S, uint32_t CG>
__global__ __launch_bounds__(kBlock) void sdpa_fold_kernel(const S *__restrict__ q,
                                                           const S *__restrict__ k,
                                                           const S *__restrict__ v,
                                                           const S *__restrict__ mask,
                                                           S *__restrict__ out, SdpaArgs a,
                                                           uint32_t parts) {
    constexpr bool kHalf = sizeof(S) == 2;
    constexpr uint32_t kAhead = 8, PL = kBlock / CG;
    __shared__ f32x4 lds_o[PL][CG];
    __shared__ f32x4 lds_ml[PL];
    const size_t rows = (size_t)a.batch * a.qh * a.ql, row = blockIdx.x;
    const uint32_t c = threadIdx.x % CG, pl = threadIdx.x / CG;
    const uint32_t d = min(4 * c, a.vdim - 4);   // columns past the end repeat the last
    const float neg_inf = -__builtin_inff();
    auto power = [](float x) { return kHalf ? __builtin_amdgcn_exp2f(x) : expf(x); };
    // the weight of a part whose maximum is m against `big`: 0 where the part
    // saw nothing, or where the row's maximum is not finite (a zero row)
    auto weight = [&](float m, float big) {
        return m == neg_inf || !__builtin_isfinite(big) ? 0.0f : power(m - big);
    };
    float big = neg_inf, total = 0.0f;
    bool nan = false;
    f32x4 acc = {0, 0, 0, 0};
    for (uint32_t p0 = pl; p0 < parts; p0 += kAhead * PL) {
        f32x4 ml[kAhead], po[kAhead];
#pragma unroll
        for (uint32_t u = 0; u < kAhead; ++u) {
            const size_t at = (size_t)min(p0 + u * PL, parts - 1) * rows + row;
            ml[u] = a.part_ml[at];
            po[u] = *reinterpret_cast<const f32x4 *>(a.part_o + at * a.vdim + d);
        }
        float now = big;
#pragma unroll
        for (uint32_t u = 0; u < kAhead; ++u)
            if (p0 + u * PL < parts) now = fmaxf(now, ml[u].x);
        const float keep = weight(big, now);
        total *= keep;
        acc *= keep;
#pragma unroll
        for (uint32_t u = 0; u < kAhead; ++u) {
            if (p0 + u * PL >= parts) continue;
            const float w = weight(ml[u].x, now);
            total += w * ml[u].y;
            acc += w * po[u];
            nan = nan || ml[u].z != 0.0f;
        }
        big = now;
    }
    lds_o[pl][c] = acc;
    if (c == 0) lds_ml[pl] = f32x4{big, total, nan ? 1.0f : 0.0f, 0.0f};
    __syncthreads();
    if (threadIdx.x >= kWave) return;   // the first wave holds every column
    big = neg_inf;
#pragma unroll
    for (uint32_t i = 0; i < PL; ++i) big = fmaxf(big, lds_ml[i].x);
    total = 0.0f;
    nan = false;
    acc = f32x4{0, 0, 0, 0};
#pragma unroll
    for (uint32_t i = 0; i < PL; ++i) {
        const f32x4 ml = lds_ml[i];
        const float w = weight(ml.x, big);
        total += w * ml.y;
        acc += w * lds_o[i][c];
        nan = nan || ml.z != 0.0f;
    }
    const bool finite = __builtin_isfinite(big), live = threadIdx.x < CG && 4 * c < a.vdim;
    const float inverse = total == 0.0f ? 0.0f : 1.0f / total;
    S res[4] __attribute__((aligned(16)));
    float odd = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        res[j] = (S)(!finite ? 0.0f : nan ? __builtin_nanf("") : acc[j] * inverse);
        odd = __builtin_fmaf(0.0f, acc[j], odd);
    }
    S *orow = out + row * a.vdim + d;
    if (live) {
        if constexpr (kHalf) *reinterpret_cast<u32x2 *>(orow) = *reinterpret_cast<const u32x2 *>(res);
        else *reinterpret_cast<u32x4 *>(orow) = *reinterpret_cast<const u32x4 *>(res);
    }
    if (__builtin_amdgcn_ballot_w64(live && finite && !nan && odd != 0.0f && __builtin_isfinite(total)) != 0) {
        __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);   // the stores above come first
        sdpa_row<S, true>(q, k, v, mask, out, a, row, threadIdx.x);
    }
}

template <typename S, int KC, int VE, int VC>
hipError_t launch_dim(const DecodePlan &p, const S *q, const S *k, const S *v, const S *mask, S *out,
                      const SdpaArgs &a, hipStream_t s) {
    const dim3 grid(a.batch * a.kvh * p.row_groups * p.parts), block(kDecodeWaves * kWave);
    const DecodeArgs da{p.parts, p.row_groups};
    if (mask)
        hipLaunchKernelGGL((sdpa_decode_kernel<S, KC, VE, VC, true>), grid, block, 0, s, q, k, v, mask, out,
                           a, da);
    else
        hipLaunchKernelGGL((sdpa_decode_kernel<S, KC, VE, VC, false>), grid, block, 0, s, q, k, v, mask, out,
                           a, da);
    return hipGetLastError();
}

template <typename S>
hipError_t fold(const DecodePlan &p, const S *q, const S *k, const S *v, const S *mask, S *out,
                const SdpaArgs &a, hipStream_t s) {
    const dim3 grid(a.batch * a.qh * a.ql), block(kBlock);
    const uint32_t groups = a.vdim / 4;
    if (groups <= 16)
        hipLaunchKernelGGL((sdpa_fold_kernel<S, 16>), grid, block, 0, s, q, k, v, mask, out, a, p.parts);
    else if (groups <= 32)
        hipLaunchKernelGGL((sdpa_fold_kernel<S, 32>), grid, block, 0, s, q, k, v, mask, out, a, p.parts);
    else
        hipLaunchKernelGGL((sdpa_fold_kernel<S, 64>), grid, block, 0, s, q, k, v, mask, out, a, p.parts);
    return hipGetLastError();
}

}  // namespace

// Which calls take the decode kernels, and how many parts the keys are cut
// into. Up to 16 packed rows always; up to 64 where packing saves blocks of
// work against the flash kernels, which give every query head its own (units:
// kv heads x row groups here, query heads there), or f32 leaves the chip
// mostly idle either way. Measured (us, flash -> here): 4 x 32q/8kv 8 x 2048
// D 128 f16 22.8 -> 18.5, 2 x 32q/4kv 8 x 4096 23.7 -> 17.0, f32 4 x 32q/8kv 16
// x 2048 87 -> 50, 12 x 24 x 2048 47.5 -> 19.3; excluded, f16 4 x 32q/8kv 16
// x 2048 23.3 vs 27.3, 8 x 12 x 24 x 600 14.1 vs 22.5, f32 35.0 vs 36.3. Where no
// heads share a kv head, f16 calls of dims 64 and 128 over long ranges are a
// little faster there (4 x 8 heads 16 x 2048 D 128 13.1 vs 15.6, 64 x 8 heads 1 x
// 2048 D 64 41.5 vs 44.7); they stay here for their P, an f16 pair instead of one f16
// (relative error of the outputs 2.0e-4, there 2.9e-4).
DecodePlan decode_plan(const k::SdpaShape &sh, bool aligned, bool f32, bool causal) {
    DecodePlan p;
    const size_t e = f32 ? 4 : 8, wide = sh.head_dim > sh.value_dim ? sh.head_dim : sh.value_dim;
    if (!aligned || !sh.batch || !sh.q_heads || !sh.kv_heads || sh.q_heads % sh.kv_heads != 0 || !sh.q_len ||
        !sh.kv_len || sh.kv_len > 0x7fffff00u || sh.head_dim == 0 || sh.value_dim == 0 ||
        sh.head_dim % e != 0 || sh.value_dim % e != 0 || wide > 256)
        return p;
    constexpr size_t kMostBlocks = 0xffffff;   // 256 work-items each
    const size_t heads = sh.batch * sh.kv_heads;
    if (sh.q_len > 64 || sh.q_heads / sh.kv_heads > 64 || heads > kMostBlocks / 4) return p;
    const size_t rows = sh.q_heads / sh.kv_heads * sh.q_len;
    if (rows > 64 || heads * rows > kMostBlocks) return p;
    p.row_groups = (uint32_t)((rows + 15) / 16);
    const size_t blocks = heads * p.row_groups;
    if (rows > 16 && 4 * blocks > 3 * sh.batch * sh.q_heads && !(f32 && blocks <= 128)) return p;
    const uint32_t tile = f32 ? 16 : 32;
    const size_t offset = sh.kv_len > sh.q_len ? sh.kv_len - sh.q_len : 0;
    const size_t seen = causal && sh.q_len + offset < sh.kv_len ? sh.q_len + offset : sh.kv_len;
    const size_t tiles = (seen + tile - 1) / tile;
    // Parts: two blocks per CU, of at least one tile per wave; the keys stay
    // whole where the second launch costs more than it spreads: K of at most
    // 80 KB per head (8 kv heads, D 64, 512 keys 6.4 us against 8.4 in parts),
    // a block per CU already (32 x 8 kv heads, 2048 keys, D 128 41.3 against
    // 45.7 in two parts), or half as many and few tiles (24 x 8 kv heads, 600
    // keys 14.2 against 17.9).
    const size_t want = (512 + blocks - 1) / blocks, fit = (tiles + 3) / 4;
    p.parts = (uint32_t)(want < fit ? want : fit);
    if (seen * sh.head_dim * (f32 ? 4 : 2) <= 80 * 1024 || blocks >= 256 || (blocks >= 128 && tiles <= 32) ||
        p.parts < 1)
        p.parts = 1;
    p.use = true;
    return p;
}

size_t decode_workspace(const DecodePlan &p, const k::SdpaShape &sh) {
    return p.parts > 1 ? (size_t)p.parts * sh.batch * sh.q_heads * sh.q_len * (sh.value_dim + 4) * sizeof(float) : 0;
}

hipError_t launch_decode_f16(const DecodePlan &p, const _Float16 *q, const _Float16 *k, const _Float16 *v,
                             const _Float16 *mask, _Float16 *out, const SdpaArgs &a, hipStream_t s) {
    const uint32_t wide = a.dim > a.vdim ? a.dim : a.vdim;
    const hipError_t e = wide <= 64    ? launch_dim<_Float16, 2, 4, 1>(p, q, k, v, mask, out, a, s)
                         : wide <= 96  ? launch_dim<_Float16, 3, 8, 1>(p, q, k, v, mask, out, a, s)
                         : wide <= 128 ? launch_dim<_Float16, 4, 8, 1>(p, q, k, v, mask, out, a, s)
                                       : launch_dim<_Float16, 8, 8, 2>(p, q, k, v, mask, out, a, s);
    return e != hipSuccess || p.parts == 1 ? e : fold<_Float16>(p, q, k, v, mask, out, a, s);
}

hipError_t launch_decode_f32(const DecodePlan &p, const float *q, const float *k, const float *v,
                             const float *mask, float *out, const SdpaArgs &a, hipStream_t s) {
    const uint32_t wide = a.dim > a.vdim ? a.dim : a.vdim;
    const hipError_t e = wide <= 64    ? launch_dim<float, 4, 4, 1>(p, q, k, v, mask, out, a, s)
                         : wide <= 128 ? launch_dim<float, 8, 4, 2>(p, q, k, v, mask, out, a, s)
                                       : launch_dim<float, 16, 4, 4>(p, q, k, v, mask, out, a, s);
    return e != hipSuccess || p.parts == 1 ? e : fold<float>(p, q, k, v, mask, out, a, s);
}

}  // namespace flash
}  // namespace icsdk
