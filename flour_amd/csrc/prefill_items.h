// prefill_items.h — the item list of the small-tile prefill kernels (device code).
#pragma once

#include <limits.h>

#include "flour_common.h"

namespace flour {

// Items of a packed batch of up to 64 sequences, longest first: an item's cost goes with the kv
// range that its rows see. BY_KV: the list goes down by levels of tile_rows positions; at level n
// stands the query tile of each sequence whose first row sees n tile_rows positions and up, its
// cached ones counted, in the order of the sequences, then `per_row` head groups of each. Without it
// levels are tile indices: the same order where no sequence has a cached prefix, and cheaper, for
// batches of one item per workgroup.
// Every wave walks the list by itself, one sequence per lane, with ballots and no barrier; BY_KV
// keeps the sequences in LDS between items (its kernel has no registers left at head_dim 128).
// A grid of G workgroups takes the list as a snake (deal), which balances it without shared
// state where the cost of item n falls with n.
struct ItemSeq {  // a sequence: first row, rows, kv length
    int c0, rows, kv;
    int at;  // BY_KV: the level of its tile 0; else its query tiles
};

template <bool BY_KV>
struct ItemWalk {
    ItemSeq mine;   // the lane's sequence
    ItemSeq* seqs;  // BY_KV: all 64, in LDS
    int shift, n_tiles, per_row;
    int level, base;  // base: items of the levels above `level`
    uint64_t there;   // sequences with a tile at `level`

    // tile_rows: a power of two; BY_KV: called by the whole workgroup, with 64 entries of LDS
    __device__ __forceinline__ void start(const int32_t* cu_seqlens, const int32_t* kv_lens,
                                          int num_seqs, int kv_cap, int tile_rows, int n_tiles_,
                                          int per_row_, int lane, ItemSeq* lds = nullptr) {
        shift = 31 - __builtin_clz(tile_rows);
        n_tiles = n_tiles_;
        per_row = per_row_;
        base = 0;
        seqs = lds;
        mine.c0 = cu_seqlens[min(lane, num_seqs)];
        mine.rows = lane < num_seqs ? cu_seqlens[lane + 1] - mine.c0 : 0;
        mine.kv = lane < num_seqs ? min(kv_lens[lane], kv_cap) : 0;
        // from the longest item on: n_tiles comes from the caller's bound on the rows, which may lie
        // far above (one step down the empty levels is ~30 cycles: a bound of 32,768 rows on 1,000
        // took 83 us instead of 21)
        if constexpr (BY_KV) {
            mine.at = max(mine.kv - mine.rows, 0) >> shift;
            if (threadIdx.x < 64) seqs[lane] = mine;
            __syncthreads();
            down_to(INT_MAX);
        } else {
            mine.at = tiles();
            level = wave_max_i32(mine.at) - 1;
            there = members();
        }
    }
    __device__ __forceinline__ int tiles() const {
        return min((max(mine.rows, 0) + (1 << shift) - 1) >> shift, n_tiles);
    }
    __device__ __forceinline__ uint64_t members() const {
        if constexpr (BY_KV) return __ballot(level >= mine.at && level < mine.at + tiles());
        return __ballot(mine.at > level);
    }
    // BY_KV: the highest level up to `from` at which a sequence has a tile (-1: none), at once, so
    // that the gap below a long context is not walked level by level
    __device__ __forceinline__ void down_to(int from) {
        const int top = min(mine.at + tiles() - 1, from);
        level = wave_max_i32(top >= mine.at ? top : -1);
        there = members();
    }
    // the workgroup's item number in a round of G: workgroup order in even rounds, reversed in odd
    static __device__ __forceinline__ int deal(int round, int G, int wg) {
        return round * G + ((round & 1) ? G - 1 - wg : wg);
    }
    // item idx (no smaller than the last one asked for): its sequence's number and facts, its tile
    // and head group; false past the list's end
    __device__ __forceinline__ bool find(int idx, int lane, int& seq, ItemSeq& s, int& tile,
                                         int& group) {
        if constexpr (BY_KV) mine = seqs[lane];
        while (level >= 0 && idx >= base + per_row * __popcll(there)) {
            base += per_row * __popcll(there);
            level--;
            there = members();
            if (BY_KV && there == 0) down_to(level);
        }
        if (level < 0) return false;
        const int rank = (idx - base) / per_row;
        group = idx - base - rank * per_row;
        const uint64_t nth =
            __ballot(((there >> lane) & 1) && __popcll(there & ((1ull << lane) - 1)) == rank);
        seq = __ffsll((unsigned long long)nth) - 1;
        s.c0 = __builtin_amdgcn_readlane(mine.c0, seq);
        s.rows = __builtin_amdgcn_readlane(mine.rows, seq);
        s.kv = __builtin_amdgcn_readlane(mine.kv, seq);
        tile = BY_KV ? level - __builtin_amdgcn_readlane(mine.at, seq) : level;
        return true;
    }
};

// Query heads per item of four (head, 32-row block) slots: 4 or 2 where at most one slot in eight
// is left without a head, else 1.
inline int item_heads(int n_rep) {
    if (n_rep % 4 == 0 || (n_rep % 4 == 3 && n_rep > 3)) return 4;
    return n_rep % 2 == 0 ? 2 : 1;
}

}  // namespace flour
