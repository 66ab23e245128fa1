// Which work item a flash-attention workgroup takes: the order of the causal and
// variable-length grids.
//
// What the order is for.  Workgroup ids go to the 8 XCDs in turn and, inside an XCD, to its
// 4 shader engines in turn (8 CUs each), whatever the load: a workgroup waits for a CU of
// its own engine.  So besides "heaviest first" the ids that are equal mod 32 must carry
// equal work.  Measured on MI355X, dK/dV kernel, causal, 32 query / 8 key-value heads:
// sequences of 4096, 3333, 2050 tokens 598 us, with one of 1024 added (3% more work) 922 us
// -- four sequences to a row of 32 workgroups had put every block of the longest one on the
// same engine of its XCD.  In the order below the same kernel takes 597 us.
#pragma once

#include "common.hpp"
#include "kernels.hpp"

namespace wmma_amd {

// The linear workgroup id of an x by y grid (by z) with the engines of every other row of 32
// ids mirrored (the XCD is kept): where the weight falls along the ids, engine 0 is first in
// one row and last in the next.  The ids of an incomplete last row stay, and so do all where
// x, the columns of equal weight, are whole rows of 32.
__device__ __forceinline__ int64_t flash_linear_id(int64_t x, int64_t y, int64_t z = 1) {
    const int64_t id = blockIdx.x + x * (blockIdx.y + y * (z > 1 ? blockIdx.z : 0));
    return (x & 31) && (id & 32) && (id | 31) < x * y * z ? id ^ 24 : id;
}

// id = row * f.d + col.
__device__ __forceinline__ int64_t flash_split_id(int64_t id, const FastDiv& f, int* col) {
    if ((id >> 31) == 0) {
        const int r = div_by(f, (int)id);
        *col = (int)((uint32_t)id - (uint32_t)r * f.d);
        return r;
    }
    const int64_t r = id / f.d;
    *col = (int)(id - r * f.d);
    return r;
}

// Strides of an attention tensor in 16-byte chunks (they are multiples of 8 elements): head
// and row fit 32 bits, so an address is a few scalar multiplies.
struct ChunkStrides {
    uint64_t batch;
    uint32_t head, row;
    // Elements to row `r` of head h of batch entry b.
    __device__ __forceinline__ int64_t at(int b, int h, int r) const {
        return (int64_t)((batch * (uint32_t)b + (uint64_t)head * (uint32_t)h +
                          (uint64_t)row * (uint32_t)r) * 8);
    }
    __device__ __forceinline__ int row_elems() const { return (int)(row * 8); }
};
inline ChunkStrides chunks_of(const AttnStrides& s) {
    return {(uint64_t)s.batch / 8, (uint32_t)(s.head / 8), (uint32_t)(s.row / 8)};
}

// Inclusive prefix sum over the 64 lanes (DPP: no LDS, no memory).
__device__ __forceinline__ int wave_scan_add(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast:15 -> rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast:31 -> rows 2, 3
    return v;
}

// Length of sequence b, clamped as every varlen kernel clamps it.
__device__ __forceinline__ int varlen_len(const int* cu, int b, int total, int longest) {
    const int a = min(max(cu[b], 0), total);
    return min(min(max(cu[b + 1], a), total) - a, longest);
}

// Blocks of `owned` rows (queries, or keys for KV) of a sequence, and how many of them
// weigh at least t, the weight being the blocks of other-side rows a block walks: all of
// them, or (causal) up to its last query / from its first key on.  Falls as t grows, so
// the blocks of one weight are a run: [nb - at_least(t), nb - at_least(t + 1)) of the query
// blocks, [at_least(t + 1), at_least(t)) of the key blocks.
template <bool KV, bool CAUSAL, int BLOCK>
__host__ __device__ __forceinline__ int varlen_at_least(int owned, int other, int t) {
    const int nb = (owned + BLOCK - 1) / BLOCK, w = (other + BLOCK - 1) / BLOCK;
    if (t <= 0) return nb;
    if (t > w) return 0;
    if (!CAUSAL) return nb;
    return KV ? min(nb, w - t + 1) : max(0, nb - (t - 1));
}

// Item `idx` of a variable-length batch, heaviest first over all of its sequences: the
// sequence b and its block.  False past the last item.  Every lane of the wave calls it
// with the same arguments (one lane per sequence, 64 at a time) and gets the same answer;
// about 0.4 us.
template <bool KV, bool CAUSAL, int BLOCK>
__device__ __forceinline__ bool varlen_item(const int* cu_q, const int* cu_k, int B, int total_q,
                                            int total_k, int max_q, int max_k, int64_t idx64,
                                            int* b_out, int* blk_out) {
    const int lane = threadIdx.x & 63;
    if (idx64 > 0x7fffffff) return false;
    const int idx = __builtin_amdgcn_readfirstlane((int)idx64);
    auto lens = [&](int b, int& owned, int& other) {
        owned = other = 0;
        if (b < B) {
            const int sq = varlen_len(cu_q, b, total_q, max_q);
            const int sk = varlen_len(cu_k, b, total_k, max_k);
            owned = KV ? sk : sq;
            other = KV ? sq : sk;
        }
    };
    int owned0, other0;  // the first 64 sequences stay in registers
    lens(lane, owned0, other0);
    auto count = [&](int t) {
        int n = varlen_at_least<KV, CAUSAL, BLOCK>(owned0, other0, t);
        for (int c = 64; c < B; c += 64) {
            int owned, other;
            lens(c + lane, owned, other);
            n += varlen_at_least<KV, CAUSAL, BLOCK>(owned, other, t);
        }
        return __builtin_amdgcn_readlane(wave_scan_add(n), 63);
    };
    if (idx >= count(0)) return false;
    // The largest weight t that more than idx items reach; `above` items weigh more.
    int lo = 0, hi = ((KV ? max_q : max_k) + BLOCK - 1) / BLOCK + 1, above = 0;
    while (hi - lo > 1) {
        const int mid = (lo + hi) / 2, n = count(mid);
        if (n > idx) {
            lo = mid;
        } else {
            hi = mid;
            above = n;
        }
    }
    int rank = idx - above;
    for (int c = 0; c < B; c += 64) {
        int owned = owned0, other = other0;
        if (c > 0) lens(c + lane, owned, other);
        const int all = varlen_at_least<KV, CAUSAL, BLOCK>(owned, other, lo);
        const int more = varlen_at_least<KV, CAUSAL, BLOCK>(owned, other, hi);
        const int upto = wave_scan_add(all - more);
        const int n = __builtin_amdgcn_readlane(upto, 63);
        if (rank < n) {
            const uint64_t reach = __builtin_amdgcn_ballot_w64(upto > rank);
            const int l = __builtin_ctzll(reach);
            const int m = rank - __builtin_amdgcn_readlane(upto - (all - more), l);
            const int nb = (__builtin_amdgcn_readlane(owned, l) + BLOCK - 1) / BLOCK;
            const int skip = __builtin_amdgcn_readlane(more, l);
            *b_out = c + l;
            *blk_out = KV ? skip + m : nb - 1 - skip - m;
            return true;
        }
        rank -= n;
    }
    return false;
}

// Whether a varlen grid of B sequences by `heads`, `blocks` per longest sequence and `parts`
// workgroups per block takes its items in that order.  Where every workgroup has a CU at once
// the search would be a visible part of them (eight sequences of 33 to 966 tokens, 8 heads: 32.6
// us in plain order, 33.2 searched; five of at most 322, 40 heads: 21.1 and 21.8).  The parts
// count: 16 / 2 heads, 1885, 2714, 371 and 949 tokens in 3 parts are 528 ids, the longest
// sequence's on one XCD (dK/dV 584 us in plain order, 246 in this one).
// The search takes about 0.5 us for 64 sequences and 0.4 for every 64 more, of every workgroup:
// only where the longest sequence has blocks enough for it.  40 heads, D = 64, forward in plain
// order and searched: 100 sequences of 16 to 200 tokens 83 and 101 us, 256 of 100 to 520 694 and
// 841, 600 of at most 371 667 and 1406; on this side of the line 64 of 300 to 760 398 and 399, 65
// of 200 to 1500 637 and 624, 16 of 400 to 3000 566 and 502 (backward 1888 and 1421).
// Whole rows of 32 heads load the engines evenly as they are.  With a causal mask, where the
// plain grid goes heaviest block first too, the search then only costs: 32 and 64 heads, D = 64
// and 128, 20 batches of 3 to 40 sequences, forward 2% and backward 1% slower searched (six of
// 100 to 2000 tokens: 56.9 and 59.1 us), none more than 3% faster.  Without one it pays but for the
// fewest sequences (32 heads, D = 64, 1945 and 276 tokens: forward 61 us in plain order, 67
// searched; three of 500 to 4000 109 and 111): over eleven batches of 4 to 24 the forward took 0
// to 15% less searched.
inline bool varlen_ordered(int64_t B, int64_t heads, int64_t blocks, int64_t parts, bool causal) {
    if (heads % 32 == 0 && (causal || B < 4)) return false;
    const int64_t passes = (B + 63) / 64;  // 64 sequences each
    return blocks >= (passes == 1 ? 3 : 2 * passes) && B * heads * blocks * parts > 256;
}

// Workgroups that a varlen grid needs for its items: no more than max_len / block per
// sequence, and no more than the packed rows hold (every sequence rounds up once).  The
// grid keeps x = B * heads, so it is never larger than one block row per max_len / block.
inline int varlen_grid_y(int64_t B, int64_t total, int64_t max_len, int64_t block) {
    const int64_t per_seq = (max_len + block - 1) / block;
    const int64_t items = B * per_seq < total / block + B ? B * per_seq : total / block + B;
    return B > 0 ? (int)((items + B - 1) / B) : 0;
}

}  // namespace wmma_amd
