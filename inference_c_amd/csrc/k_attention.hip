// Scaled dot-product attention for gfx950, with the accelerator semantics of
// the reference's attention backends (src/platform/cuda/attention_cuda.cu:
// 25-99):
//     s[j]   = (sum over d, in order, of q[d] k[j][d]) * scale (+ mask[i][j]),
//              -inf where causal and j > i + (kv_len - q_len);
//     a row whose maximum score (NaN ignored) is not finite is all zeros;
//     p[j]   = exp(s[j] - max) / sum_j exp(s[j] - max);
//     out[e] = sum_j p[j] v[j][e].
// q [B, Hq, Lq, D], k [B, Hkv, Lkv, D], v [B, Hkv, Lkv, Dv], mask [Lq, Lkv],
// out [B, Hq, Lq, Dv]; query head h reads kv head h / (Hq / Hkv).
//
// Row kernel (any D, Dv up to 512; f32 and f16): one wave per query row,
// keys in chunks of 64 with the running max and sum of an online softmax.
// Within a chunk, lane j owns key j: it forms the score as a sequential f32
// dot product (the same order and roundings as the reference, so scores are
// bit-identical), the wave folds the chunk into the running max and sum, and
// then lane e owns output element e (+64, +128, ...) and accumulates
// p[j] * v[j][e] over the chunk, reading p[j] and q[d] from the owning lane
// with v_readlane. No LDS and no barriers. The weights are normalised once at
// the end (acc / sum) rather than per weight, and the online rescaling
// reorders the roundings of p; outputs therefore agree with the reference to
// a few roundings of sum_j p_j |v_j|.
#include "decode.hpp"
#include "flash.hpp"
#include "kern_common.hpp"
#include "kernels.hpp"
#include "sdk.hpp"

#include <algorithm>

namespace icsdk {
namespace {

using namespace flash;

template <typename S, bool kVec>
__global__ __launch_bounds__(kBlock) void sdpa_row_kernel(const S *__restrict__ q,
                                                          const S *__restrict__ k,
                                                          const S *__restrict__ v,
                                                          const S *__restrict__ mask,
                                                          S *__restrict__ out, SdpaArgs a) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const size_t row = (size_t)blockIdx.x * (kBlock / kWave) +
                       (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    if (row >= (size_t)a.batch * a.qh * a.ql) return;
    sdpa_row<S, kVec>(q, k, v, mask, out, a, row, lane);
}

template <typename S>
hipError_t launch_sdpa(const S *q, const S *k, const S *v, const S *mask, S *out,
                       const k::SdpaShape &sh, float scale, bool causal, hipStream_t s) {
    if (sh.batch == 0 || sh.q_heads == 0 || sh.kv_heads == 0 || sh.q_len == 0 ||
        sh.kv_len == 0 || sh.head_dim == 0 || sh.value_dim == 0 ||
        sh.q_heads % sh.kv_heads != 0)
        return hipErrorInvalidValue;
    if (sh.head_dim > (size_t)kMaxRowRegs * kWave || sh.value_dim > (size_t)kMaxRowRegs * kWave)
        return hipErrorInvalidValue;
    const uint64_t lim = 0xffffffffull;
    if (sh.batch > lim || sh.q_heads > lim || sh.kv_heads > lim || sh.q_len > lim ||
        sh.kv_len > lim)
        return hipErrorInvalidValue;
    SdpaArgs a{};
    a.batch = (uint32_t)sh.batch;
    a.qh = (uint32_t)sh.q_heads;
    a.kvh = (uint32_t)sh.kv_heads;
    a.group = (uint32_t)(sh.q_heads / sh.kv_heads);
    a.ql = (uint32_t)sh.q_len;
    a.kl = (uint32_t)sh.kv_len;
    a.dim = (uint32_t)sh.head_dim;
    a.vdim = (uint32_t)sh.value_dim;
    a.causal_offset = a.kl > a.ql ? a.kl - a.ql : 0;
    a.scale = scale;
    a.causal = causal ? 1 : 0;
    const size_t rows = sh.batch * sh.q_heads * sh.q_len;
    const size_t waves_per_block = kBlock / kWave;
    const size_t blocks = (rows + waves_per_block - 1) / waves_per_block;
    if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
    constexpr size_t E = Vec16<S>::N;
    if (sh.head_dim % E == 0 && ((uintptr_t)k & 15u) == 0)
        hipLaunchKernelGGL((sdpa_row_kernel<S, true>), dim3((unsigned)blocks), dim3(kBlock), 0, s,
                           q, k, v, mask, out, a);
    else
        hipLaunchKernelGGL((sdpa_row_kernel<S, false>), dim3((unsigned)blocks), dim3(kBlock), 0,
                           s, q, k, v, mask, out, a);
    return hipGetLastError();
}

}  // namespace

namespace {

// Flash path choice for a shape: f16 256-query blocks (8 waves sharing each
// K/V tile) when there are at least 256 of them (32 x 2048^2 D 128 82.8 us
// vs 89.2 with 128-query blocks, 4096^2 causal 164.6 vs 179.9; 4 x 16 x
// 512^2, 128 such blocks, 23.5 vs 20.9), else 128-query blocks (4 waves)
// when there are at least 64 of them, else 64-query blocks (measured:
// 12 x 1024^2 D 64 f16 20.1 us wide vs 22.2 narrow, 4 x 16 x 512^2 D 128
// 21.1 vs 25.6, 32 x 1024^2 causal 33.2 vs 39.0, f32 4 x 16 x 512^2 56.6
// vs 70.6; f32 stays at 128). The work is then cut into items and ordered longest first.
// With a workspace, query blocks whose key range is long against the whole
// launch are split: target split_tiles = max(total key tiles / slots,
// kMinPartTiles), slots measured over 128 .. 3072: f16 128 (a split rarely
// pays for its merge: the vision shape is best in 2 parts, 32 x 2048^2
// causal unsplit; grids of up to 256 blocks of 128 queries take 256 and
// the parts fitted to one round, below), f32 512 (its 32-key tiles of
// 64 MFMAs keep a block busy: 12 x 1024^2 D 64 53 us in 6 parts vs 59 in
// 2 and 103 unsplit; 4 x 16 x 512^2, 256 blocks, is best unsplit). The
// part size grows until a (batch, head)'s items fit kMaxFlashItems; more
// query blocks than that: descending query blocks, no split.
struct FlashPlan {
    bool flash = false;
    uint32_t dim = 0;            // head dim the kernel is compiled for
    bool any_dim = false;        // rows narrower than `dim`, or K and V of different widths
    uint32_t bm = 64, tk = 64;   // queries per block (64, 128, or 256 for f16), keys per tile
    uint32_t key_parts = 1;      // f16: waves per query group, taking alternate key tiles
    uint32_t qblocks = 0, items = 0;
    uint32_t split_tiles = 0;
    uint32_t max_parts = 1;
    uint32_t first_split = 0;   // first split query block
    bool table = false, xcd_heads = false;
    uint32_t item[kMaxFlashItems] = {};
};

// f16 blocks of 128 queries whose 8 waves split the key tiles in two (see
// sdpa_flash_kernel) pay where a causal launch is about one round of
// 256-query blocks with uneven key ranges: twice as many blocks, each half
// as long, let the longest-first order pair long blocks with short ones on
// a CU, with no merge launch. Measured (us, two-part vs 256-query blocks):
// 32q/8kv 2048^2 D 128 causal 58.4 vs 70.3, D 64 37.3 vs 50.0; 32 x 1024^2
// D 64 causal 17.5 vs 22.4 (128-query blocks). Each two-part step stages
// twice the K/V bytes per wave, so where the key ranges are even, or there
// are several rounds of blocks for the order to balance, they lose: 2048^2
// D 128 non-causal 95 vs 80, 4096^2 causal 187 vs 167, 4 x 2048^2 causal
// 220 vs 189.
// f32: the same in-block split for causal launches of at least one 8-wave
// block per CU with uneven key ranges (measured below)
bool key_parts_pay_f32(const k::SdpaShape &sh, bool causal) {
    const size_t bhs = sh.batch * sh.q_heads;
    if (!causal || ((sh.q_len + 127) / 128) * bhs < 256) return false;
    const uint32_t ql = (uint32_t)sh.q_len, kl = (uint32_t)sh.kv_len;
    const uint32_t offset = kl > ql ? kl - ql : 0, blocks = (ql + 127) / 128;
    // every block up to 1024 of them, else an even sample (the longest,
    // the last block, always in it)
    const uint32_t stride = blocks > 1024 ? blocks / 1024 : 1;
    uint64_t total = 0, most = 0, n = 0;
    for (uint32_t j = blocks - 1;; j -= stride) {
        const uint64_t t = flash_tiles(ql, kl, true, offset, 128, kFlashN32, j);
        total += t;
        most = t > most ? t : most;
        ++n;
        if (j < stride) break;
    }
    return 4 * most * n > 5 * total;
}

bool key_parts_pay(const k::SdpaShape &sh, bool causal) {
    const size_t bhs = sh.batch * sh.q_heads;
    if (!causal || ((sh.q_len + 127) / 128) * bhs < 256 || ((sh.q_len + 255) / 256) * bhs > 256)
        return false;
    // uneven: the longest 256-query block sees > 5/4 of the average key tiles
    const uint32_t ql = (uint32_t)sh.q_len, kl = (uint32_t)sh.kv_len;
    const uint32_t offset = kl > ql ? kl - ql : 0, blocks = (ql + 255) / 256;
    uint64_t total = 0, most = 0;
    for (uint32_t j = 0; j < blocks; ++j) {
        const uint64_t t = flash_tiles(ql, kl, true, offset, 256, kFlashN, j);
        total += t;
        most = t > most ? t : most;
    }
    return 4 * most * blocks > 5 * total;
}

// The head dim a flash kernel is compiled for that serves rows of these
// widths, or 0: the kernels need every row to start on 16 bytes (whole
// vectors per row); past 256 the row kernel stays. Of the dims between, 80 and
// 96 are compiled because vision encoders use them (72 .. 96); one MFMA
// chunk of padding costs 1/5 of the score MFMAs.
uint32_t flash_dim(const k::SdpaShape &sh, bool f32) {
    const size_t e = f32 ? 4 : 8, wide = std::max(sh.head_dim, sh.value_dim);
    if (sh.head_dim % e != 0 || sh.value_dim % e != 0 || wide == 0) return 0;
    for (uint32_t d : {32u, 64u, 80u, 96u, 128u, 256u})
        if (wide <= d) return d == 64 && (sh.head_dim != 64 || sh.value_dim != 64) ? 80 : d;
    return 0;
}

FlashPlan flash_plan(const k::SdpaShape &sh, bool aligned, bool f32, bool causal, bool split) {
    FlashPlan p;
    const uint64_t lim = 0x7fffffffull;
    p.dim = flash_dim(sh, f32);
    p.any_dim = sh.head_dim != sh.value_dim || (sh.head_dim != 64 && sh.head_dim != 128);
    if (!aligned || p.dim == 0 ||
        !sh.batch || !sh.q_heads || !sh.kv_heads || sh.q_heads % sh.kv_heads != 0 ||
        !sh.q_len || sh.q_len > lim || !sh.kv_len || sh.kv_len > lim ||
        sh.batch * sh.q_heads * ((sh.q_len + 63) / 64) > lim / (8 * kMaxKeyParts))
        return p;
    p.flash = true;
    const size_t bhs = sh.batch * sh.q_heads;
    // f16 grids of 64-255 blocks of 128 queries (fewer blocks than CUs)
    // also take two key parts, with the key-range split across blocks kept:
    // twice the waves per block (12 heads x 1024^2 D 64: 18.7 -> 16.9 us).
    // Non-causal ones of at most 128 such blocks over at most 1024 keys take
    // 64-query blocks (4 waves: 2 query groups x 2 key parts) and no split:
    // at most one block per CU, no merge launch (us, same box: 12 heads x
    // 1024^2 D 64 17.4 -> 14.3, D 128 25.9 -> 20.8, 32 heads x 512^2 D 64
    // 11.2 -> 9.6, 8 heads x 1024^2 D 64 15.7 -> 13.8); over 2048 keys, or
    // with more blocks than CUs, the split plan stays faster (4 heads x
    // 2048^2 D 128 31.7 vs 35.7; 20 heads x 1024^2 D 64 17.0 vs 25.9).
    // Exactly 256 such blocks (one per CU; not the 256-query plan) likewise
    // take two key parts: 8 waves per CU instead of 4 (us, same box: 32 x
    // 1024^2 D 64 non-causal 22.8 -> 18.7, 32q/8kv 1024 x 4096 D 128 109 ->
    // 90, causal 32 x 1024 x 4096 D 64 (even key ranges) 77 -> 57; with 384
    // blocks, two rounds, they lose: 48 x 1024^2 D 64 30.1 vs 34.1).
    const uint64_t q128 = ((sh.q_len + 127) / 128) * bhs;
    const bool small_grid = !f32 && q128 >= 64 &&
                            (q128 < 256 || (q128 == 256 && ((sh.q_len + 255) / 256) * bhs < 256));
    const bool small_short = small_grid && !causal && q128 <= 128 && sh.kv_len <= 1024;
    // Grids of fewer than 64 blocks of 128 queries: 64-query blocks of 4
    // waves (2 query groups x 2 key parts), the key range split over blocks
    // as before (us, same box, one-part 64-query blocks -> two-part: f16
    // 32q/8kv 128 x 2048 D 128 causal 33.3 -> 25.3, 8 x 512 x 4096 D 128
    // causal 55.0 -> 39.7, 40q/8kv 64 x 4096 D 128 33.0 -> 25.3, 16 x 256 x
    // 1024 D 64 15.5 -> 12.5, 8 x 512^2 D 128 14.7 -> 13.5; f32 16 x 256 x
    // 1024 D 64 34.7 -> 26.1, 4 x 1024^2 D 64 32.9 -> 24.6, 8 x 512^2 D 128
    // 32.8 -> 25.1). f32 at D 128 over more keys keeps one part (its
    // two-part 64-query block needs ~300 registers, one wave per SIMD:
    // 32q/8kv 128 x 2048 63.6 vs 68.9, 8 x 512 x 4096 causal 103 vs 111).
    const bool tiny_grid = q128 < 64 && (!f32 || p.dim <= 64 || sh.kv_len <= 512);
    // one key part per query group where two do not fit: two parts of
    // 256-wide K and V tiles exceed the LDS, and the f32 kernels of other
    // dims are compiled with one
    const bool one_part = p.any_dim && (f32 || p.dim > 128);
    if (one_part) {
        p.bm = q128 >= 64 ? 128 : 64;
    } else if (f32 ? key_parts_pay_f32(sh, causal) : key_parts_pay(sh, causal)) {
        p.bm = 128;
        p.key_parts = 2;
    } else if (small_grid) {
        p.bm = small_short ? 64 : 128;
        p.key_parts = 2;
    } else if (tiny_grid) {
        p.bm = 64;
        p.key_parts = 2;
    } else if (!f32) {
        // more than 256 blocks of 128 queries: 256-query blocks, also below
        // one round of them (us, same box, 128-query blocks -> 256: 48 x
        // 1024^2 D 64 30.4 -> 29.7, 32q/8kv 1536^2 D 128 59.4 -> 58.0, causal
        // 48q/8kv 1024 x 4096 D 128 135 -> 132)
        p.bm = 256;
    } else if (q128 >= 64) p.bm = 128;
    else p.bm = 64;
    p.tk = f32 ? 32 : 64;
    p.qblocks = (uint32_t)((sh.q_len + p.bm - 1) / p.bm);
    // more work-items than a launch holds (2^23 heads of a few queries with 512
    // threads each): the row kernel
    if (bhs * p.qblocks * 2 * p.bm * p.key_parts > 0xffffffffull) return FlashPlan{};
    p.items = p.qblocks;
    p.first_split = p.qblocks;
    p.xcd_heads = (sh.batch * sh.kv_heads) % 8 == 0;
    if (p.qblocks > kMaxFlashItems) return p;
    const uint32_t ql = (uint32_t)sh.q_len, kl = (uint32_t)sh.kv_len;
    const uint32_t offset = kl > ql ? kl - ql : 0;
    auto tiles = [&](uint32_t j) { return flash_tiles(ql, kl, causal, offset, p.bm, p.tk, j); };
    // f32 launches of two key parts in one round (256 blocks of 128
    // queries) split the long blocks' key ranges as well (us, same box:
    // causal 16 x 2048^2 D 64 171 -> 135, D 128 300 -> 228); from two rounds
    // on the longest-first order balances them without the merge's traffic
    const bool f32_round_split = f32 && p.key_parts == 2 && q128 <= 256;
    if (split && (p.key_parts == 1 || (small_grid && !small_short) || tiny_grid || f32_round_split)) {
        uint64_t total = 0;
        for (uint32_t j = 0; j < p.qblocks; ++j) total += tiles(j);
        total *= bhs;
        // f16 grids of up to 256 blocks (one per CU: the two-part blocks
        // take up to 151 KB of LDS) cut their key ranges into the most
        // parts that still fit one round of 256 blocks (us, same box, 128
        // slots before: 32q/8kv decode over 16384 keys 64.5 -> 37.0, 4 x
        // 32q/8kv decode over 2048 keys 34.2 -> 22.5, 32q/8kv 16 x 4096 causal
        // 22.8 -> 16.6, 8 x 512 x 4096 causal 39.5 -> 28.3, 8 x 1024 x 8192
        // 76.7 -> 54.3, 16 x 1024 x 4096 causal 48.7 -> 37.0; others equal)
        const bool fit = !f32 && (tiny_grid || small_grid) && !one_part;
        const uint64_t slots = f32 ? 512 : fit ? 256 : 128;
        const uint64_t target = (total + slots - 1) / slots;
        p.split_tiles = (uint32_t)(target > kMinPartTiles ? target : kMinPartTiles);
        // The smallest part size from there whose items fit the work table
        // (kMaxFlashItems per (batch, head)) and, for `fit`, 256 blocks in
        // all. The item count never grows with the part size, so a binary
        // search; at the largest size every query block is one item.
        auto parts_of = [&](uint32_t st) {
            uint64_t n = 0;
            for (uint32_t j = 0; j < p.qblocks; ++j) n += split_parts(tiles(j), st);
            return n;
        };
        auto fits = [&](uint32_t st) {
            const uint64_t n = parts_of(st);
            return n <= kMaxFlashItems && (!fit || n * bhs <= 256);
        };
        uint32_t lo = p.split_tiles, hi = lo;
        for (uint32_t j = 0; j < p.qblocks; ++j) hi = tiles(j) > hi ? tiles(j) : hi;
        while (lo < hi) {
            const uint32_t mid = lo + (hi - lo) / 2;
            if (fits(mid)) hi = mid;
            else lo = mid + 1;
        }
        p.split_tiles = lo;
    }
    struct Item {
        uint32_t size, qblock, part, parts;
    };
    Item list[kMaxFlashItems];
    uint32_t n = 0;
    for (uint32_t j = 0; j < p.qblocks; ++j) {
        const uint32_t t = tiles(j), parts = split_parts(t, p.split_tiles);
        const uint32_t share = (t + parts - 1) / parts;
        if (n + parts > kMaxFlashItems) {   // too many: descending query blocks, whole
            p.split_tiles = 0;
            p.max_parts = 1;
            p.first_split = p.qblocks;
            return p;
        }
        for (uint32_t q = 0; q < parts; ++q) {
            const uint32_t lo = q * share < t ? q * share : t;
            const uint32_t hi = lo + share < t ? lo + share : t;
            list[n++] = Item{hi - lo, j, q, parts};
        }
        if (parts > p.max_parts) p.max_parts = parts;
        if (parts > 1 && j < p.first_split) p.first_split = j;
    }
    std::stable_sort(list, list + n, [](const Item &x, const Item &y) {
        return x.size != y.size ? x.size > y.size : x.qblock > y.qblock;
    });
    p.items = n;
    p.table = true;
    for (uint32_t r = 0; r < n; ++r)
        p.item[r] = list[r].qblock | list[r].part << 16 | list[r].parts << 24;
    if (p.max_parts == 1) p.split_tiles = 0;
    return p;
}

size_t partial_bytes(const k::SdpaShape &sh, uint32_t parts) {
    const size_t rows = sh.batch * sh.q_heads * sh.q_len;
    return (size_t)parts * rows * (sh.value_dim + 4) * sizeof(float);
}

// The plan for a launch: split only when the caller's workspace holds the
// partial results.
FlashPlan launch_plan(const k::SdpaShape &sh, bool aligned, bool f32, bool causal,
                      size_t workspace_bytes, const void *workspace) {
    const FlashPlan p = flash_plan(sh, aligned, f32, causal, true);
    if (p.max_parts > 1 && (workspace == nullptr || workspace_bytes < partial_bytes(sh, p.max_parts)))
        return flash_plan(sh, aligned, f32, causal, false);
    return p;
}

SdpaArgs flash_args(const FlashPlan &p, const k::SdpaShape &sh, float scale, bool causal,
                    void *workspace) {
    SdpaArgs a{};
    a.batch = (uint32_t)sh.batch;
    a.qh = (uint32_t)sh.q_heads;
    a.kvh = (uint32_t)sh.kv_heads;
    a.group = (uint32_t)(sh.q_heads / sh.kv_heads);
    a.ql = (uint32_t)sh.q_len;
    a.kl = (uint32_t)sh.kv_len;
    a.dim = (uint32_t)sh.head_dim;
    a.vdim = (uint32_t)sh.value_dim;
    a.causal_offset = a.kl > a.ql ? a.kl - a.ql : 0;
    a.scale = scale;
    a.causal = causal ? 1 : 0;
    a.items = p.items;
    a.qblocks = p.qblocks;
    a.split_tiles = p.split_tiles;
    a.table = p.table ? 1 : 0;
    a.xcd_heads = p.xcd_heads ? 1 : 0;
    for (uint32_t r = 0; r < p.items && p.table; ++r) a.item[r] = p.item[r];
    if (p.max_parts > 1) {
        const size_t rows = sh.batch * sh.q_heads * sh.q_len;
        a.part_o = static_cast<float *>(workspace);
        a.part_ml = reinterpret_cast<f32x4 *>(a.part_o + (size_t)p.max_parts * rows * sh.value_dim);
    }
    return a;
}

// The decode kernels' plan and arguments, or use == false. Without the
// workspace for several parts the keys stay in one.
DecodePlan decode_args(const k::SdpaShape &sh, bool aligned, bool f32, float scale, bool causal,
                       void *workspace, size_t workspace_bytes, SdpaArgs *a) {
    DecodePlan d = decode_plan(sh, aligned, f32, causal);
    if (!d.use) return d;
    if (d.parts > 1 && (workspace == nullptr || workspace_bytes < decode_workspace(d, sh))) d.parts = 1;
    *a = flash_args(FlashPlan{}, sh, scale, causal, nullptr);
    if (d.parts > 1) {
        a->part_o = static_cast<float *>(workspace);
        a->part_ml = reinterpret_cast<f32x4 *>(a->part_o + (size_t)d.parts * sh.batch * sh.q_heads * sh.q_len * sh.value_dim);
    }
    return d;
}

template <typename S, bool kAnyDim>
hipError_t combine_splits(const SdpaArgs &a, const FlashPlan &p, const S *q, const S *k, const S *v,
                          const S *mask, S *out, hipStream_t s) {
    const uint32_t first_row = p.first_split * p.bm;
    const size_t n = (size_t)a.batch * a.qh * (a.ql - first_row) * combine_lanes<S, kAnyDim>(a.vdim);
    const dim3 grid((unsigned)((n + kBlock - 1) / kBlock)), block(kBlock);
    // the part-count bucket: no row of this launch has more parts
    static_assert(kMaxKeyParts <= 8, "combine buckets");
    if (p.max_parts <= 2)
        hipLaunchKernelGGL((sdpa_combine_kernel<S, sizeof(S) == 2, 2, kAnyDim>), grid, block, 0, s,
                           a, out, p.bm, p.tk, first_row, q, k, v, mask);
    else if (p.max_parts <= 4)
        hipLaunchKernelGGL((sdpa_combine_kernel<S, sizeof(S) == 2, 4, kAnyDim>), grid, block, 0, s,
                           a, out, p.bm, p.tk, first_row, q, k, v, mask);
    else
        hipLaunchKernelGGL((sdpa_combine_kernel<S, sizeof(S) == 2, 8, kAnyDim>), grid, block, 0, s,
                           a, out, p.bm, p.tk, first_row, q, k, v, mask);
    return hipGetLastError();
}

}  // namespace

// One flash launch for the plan's (D, BM, KS) with the general (mask) /
// split variant.
#define ICSDK_FLASH_VARIANTS_KS(KERNEL, D, BM, KS, Q, K, V, M, O)                                  \
    do {                                                                                           \
        if (general && split)                                                                      \
            hipLaunchKernelGGL((KERNEL<D, BM, true, true, KS>), grid, block, 0, s, Q, K, V, M, O, a);  \
        else if (general)                                                                          \
            hipLaunchKernelGGL((KERNEL<D, BM, true, false, KS>), grid, block, 0, s, Q, K, V, M, O, a); \
        else if (split)                                                                            \
            hipLaunchKernelGGL((KERNEL<D, BM, false, true, KS>), grid, block, 0, s, Q, K, V, M, O, a); \
        else                                                                                       \
            hipLaunchKernelGGL((KERNEL<D, BM, false, false, KS>), grid, block, 0, s, Q, K, V, M, O, a);\
    } while (0)
// two-part blocks of 64 or 128 queries
#define ICSDK_FLASH_VARIANTS_KS2_BM(KERNEL, D, Q, K, V, M, O)                                     \
    do {                                                                                           \
        if (plan.bm == 64) ICSDK_FLASH_VARIANTS_KS(KERNEL, D, 64, 2, Q, K, V, M, O);               \
        else ICSDK_FLASH_VARIANTS_KS(KERNEL, D, 128, 2, Q, K, V, M, O);                            \
    } while (0)
// the f32 kernel: 64- or 128-query blocks, 64- or 128-query blocks with two
// key parts per query group
#define ICSDK_FLASH_SHAPES_F32(KERNEL, Q, K, V, M, O)                                              \
    do {                                                                                           \
        if (shape.head_dim == 64) {                                                                \
            if (ks == 2) ICSDK_FLASH_VARIANTS_KS2_BM(KERNEL, 64, Q, K, V, M, O);                   \
            else if (plan.bm == 128) ICSDK_FLASH_VARIANTS_KS(KERNEL, 64, 128, 1, Q, K, V, M, O);   \
            else ICSDK_FLASH_VARIANTS_KS(KERNEL, 64, 64, 1, Q, K, V, M, O);                        \
        } else {                                                                                   \
            if (ks == 2) ICSDK_FLASH_VARIANTS_KS2_BM(KERNEL, 128, Q, K, V, M, O);                  \
            else if (plan.bm == 128) ICSDK_FLASH_VARIANTS_KS(KERNEL, 128, 128, 1, Q, K, V, M, O);  \
            else ICSDK_FLASH_VARIANTS_KS(KERNEL, 128, 64, 1, Q, K, V, M, O);                       \
        }                                                                                          \
    } while (0)
// the f16 kernel: 64-, 128- or 256-query blocks, 64- or 128-query blocks
// with two key parts per query group
#define ICSDK_FLASH_SHAPES_F16(KERNEL, Q, K, V, M, O)                                              \
    do {                                                                                           \
        const int bm = (int)plan.bm;                                                               \
        if (shape.head_dim == 64) {                                                                \
            if (ks == 2) ICSDK_FLASH_VARIANTS_KS2_BM(KERNEL, 64, Q, K, V, M, O);                      \
            else if (bm == 256) ICSDK_FLASH_VARIANTS_KS(KERNEL, 64, 256, 1, Q, K, V, M, O);        \
            else if (bm == 128) ICSDK_FLASH_VARIANTS_KS(KERNEL, 64, 128, 1, Q, K, V, M, O);        \
            else ICSDK_FLASH_VARIANTS_KS(KERNEL, 64, 64, 1, Q, K, V, M, O);                        \
        } else {                                                                                   \
            if (ks == 2) ICSDK_FLASH_VARIANTS_KS2_BM(KERNEL, 128, Q, K, V, M, O);                     \
            else if (bm == 256) ICSDK_FLASH_VARIANTS_KS(KERNEL, 128, 256, 1, Q, K, V, M, O);       \
            else if (bm == 128) ICSDK_FLASH_VARIANTS_KS(KERNEL, 128, 128, 1, Q, K, V, M, O);       \
            else ICSDK_FLASH_VARIANTS_KS(KERNEL, 128, 64, 1, Q, K, V, M, O);                       \
        }                                                                                          \
    } while (0)

namespace k {

// An output in place of q keeps off the kernels that may do a row again, which
// reads its q a second time: the decode kernels, and the f16 flash kernels of
// other head dims than 64 and 128.
//
// A call that a graph records takes the same kernels as one that runs. At D 64
// and 128 its key parts hold memory of the graph's own; at other head dims the
// keys stay in one part, so such a graph holds one kernel and no memory
// (decode kernels with one part against flash kernels with one, us: f16 32q/8kv
// over 2048 keys D 128 22 against 33, 16q/4kv D 80 26 against 32, f32 59
// against 238; never slower at 16 shapes of either type).
size_t sdpa_workspace_bytes(const SdpaShape &shape, bool f32, bool causal, const void *q,
                            const void *out) {
    const bool in_place = q == out;
    const bool whole_dims = shape.head_dim == shape.value_dim && (shape.head_dim == 64 || shape.head_dim == 128);
    if (!whole_dims && sdk_recording() != Recording::kNo) return 0;
    const DecodePlan d = decode_plan(shape, !in_place, f32, causal);
    if (d.use) return decode_workspace(d, shape);
    const FlashPlan p = flash_plan(shape, true, f32, causal, true);
    if (!p.flash || p.max_parts == 1 || (in_place && p.any_dim && !f32)) return 0;
    return partial_bytes(shape, p.max_parts);
}

hipError_t sdpa_f32(const float *q, const float *k, const float *v, const float *mask,
                    float *out, const SdpaShape &shape, float scale, bool causal,
                    void *workspace, size_t workspace_bytes, hipStream_t s) {
    const bool aligned = (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15u) == 0;
    SdpaArgs da;
    const DecodePlan decode = decode_args(shape, aligned && q != out, true, scale, causal, workspace,
                                          workspace_bytes, &da);
    if (decode.use) return launch_decode_f32(decode, q, k, v, mask, out, da, s);
    const FlashPlan plan = launch_plan(shape, aligned, true, causal, workspace_bytes, workspace);
    if (!plan.flash) return launch_sdpa<float>(q, k, v, mask, out, shape, scale, causal, s);
    const SdpaArgs a = flash_args(plan, shape, scale, causal, workspace);
    const bool split = plan.max_parts > 1;
    const bool general = mask != nullptr;
    // with a mask a second key part pays from the second key tile on (its
    // clamped mask loads cost more than a plain tile's: 16 x 8 heads 50 x 50
    // D 64 f16 6.5 us, two parts 8.2)
    const uint32_t ks = general && shape.kv_len <= plan.tk ? 1 : plan.key_parts;
    const dim3 grid((unsigned)(shape.batch * shape.q_heads * plan.items)), block(2 * plan.bm * ks);
    if (plan.any_dim) {
        const hipError_t status = launch_any_dim_f32({plan.dim, plan.bm, ks, general, split}, grid,
                                                     block, s, q, k, v, mask, out, a);
        return status != hipSuccess || !split ? status : combine_splits<float, true>(a, plan, q, k, v, mask, out, s);
    }
    ICSDK_FLASH_SHAPES_F32(sdpa_flash_f32_kernel, q, k, v, mask, out);
    const hipError_t status = hipGetLastError();
    return status != hipSuccess || !split ? status : combine_splits<float, false>(a, plan, q, k, v, mask, out, s);
}

hipError_t sdpa_f16(const uint16_t *q, const uint16_t *k, const uint16_t *v,
                    const uint16_t *mask, uint16_t *out, const SdpaShape &shape, float scale,
                    bool causal, void *workspace, size_t workspace_bytes, hipStream_t s) {
    auto h = [](const uint16_t *p) { return reinterpret_cast<const _Float16 *>(p); };
    _Float16 *o16 = reinterpret_cast<_Float16 *>(out);
    const bool aligned = (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15u) == 0;
    SdpaArgs da;
    const DecodePlan decode = decode_args(shape, aligned && q != out, false, scale, causal, workspace,
                                          workspace_bytes, &da);
    if (decode.use) return launch_decode_f16(decode, h(q), h(k), h(v), h(mask), o16, da, s);
    const FlashPlan plan = launch_plan(shape, aligned, false, causal, workspace_bytes, workspace);
    if (!plan.flash || (plan.any_dim && q == out))
        return launch_sdpa<_Float16>(h(q), h(k), h(v), h(mask), o16, shape, scale, causal, s);
    const SdpaArgs a = flash_args(plan, shape, scale, causal, workspace);
    const bool split = plan.max_parts > 1;
    // the raw-product softmax needs scale > 0; other scales take the general
    // (mask) variant, whose mask may be null
    const bool general = mask != nullptr || !(scale > 0.0f);
    const uint32_t ks = general && shape.kv_len <= plan.tk ? 1 : plan.key_parts;
    const dim3 grid((unsigned)(shape.batch * shape.q_heads * plan.items)), block(2 * plan.bm * ks);
    if (plan.any_dim) {
        const hipError_t status = launch_any_dim_f16({plan.dim, plan.bm, ks, general, split}, grid,
                                                     block, s, h(q), h(k), h(v), h(mask), o16, a);
        return status != hipSuccess || !split ? status : combine_splits<_Float16, true>(a, plan, h(q), h(k), h(v), h(mask), o16, s);
    }
    ICSDK_FLASH_SHAPES_F16(sdpa_flash_kernel, h(q), h(k), h(v), h(mask), o16);
    const hipError_t status = hipGetLastError();
    return status != hipSuccess || !split ? status : combine_splits<_Float16, false>(a, plan, h(q), h(k), h(v), h(mask), o16, s);
}

}  // namespace k

#undef ICSDK_FLASH_SHAPES_F16
#undef ICSDK_FLASH_SHAPES_F32
#undef ICSDK_FLASH_VARIANTS_KS2_BM
#undef ICSDK_FLASH_VARIANTS_KS

}  // namespace icsdk
