// prefill_items.h — the item list of the small-tile prefill kernels (device code).
#pragma once

#include "flour_common.h"

namespace flour {

// Items of a packed batch of up to 64 sequences, longest first: query tiles by decreasing tile
// index (a tile's causal kv range grows with it), then sequences, then `per_row` head groups.
// Every wave walks the list by itself, one sequence per lane, with ballots: no LDS, no barrier.
// A grid of G workgroups takes the list as a snake (deal), which balances it without shared
// state: the cost of item n falls with n.
struct ItemWalk {
    int c0, rows, kv, tiles;  // the lane's sequence: first row, rows, kv length, query tiles
    int per_row, level, base;  // items of the levels above `level`
    uint64_t there;            // sequences with a tile at `level`

    __device__ __forceinline__ void start(const int32_t* cu_seqlens, const int32_t* kv_lens,
                                          int num_seqs, int kv_cap, int tile_rows, int n_tiles,
                                          int per_row_, int lane) {
        c0 = cu_seqlens[min(lane, num_seqs)];
        rows = lane < num_seqs ? cu_seqlens[lane + 1] - c0 : 0;
        kv = lane < num_seqs ? min(kv_lens[lane], kv_cap) : 0;
        tiles = rows > 0 ? (rows + tile_rows - 1) / tile_rows : 0;
        per_row = per_row_;
        // from the longest sequence on: n_tiles comes from the caller's bound on the rows, which may
        // lie far above (one step down the empty levels is ~30 cycles: a bound of 32,768 rows on
        // 1,000 took 83 us instead of 21)
        level = min(n_tiles, __builtin_amdgcn_readfirstlane((int)wave_max((float)tiles))) - 1;
        base = 0;
        there = __ballot(tiles > level);
    }
    // the workgroup's item number in a round of G: workgroup order in even rounds, reversed in odd
    static __device__ __forceinline__ int deal(int round, int G, int wg) {
        return round * G + ((round & 1) ? G - 1 - wg : wg);
    }
    // item idx (no smaller than the last one asked for): its sequence, tile and head group; false
    // past the list's end
    __device__ __forceinline__ bool find(int idx, int lane, int& seq, int& tile, int& group) {
        while (level >= 0 && idx >= base + per_row * __popcll(there)) {
            base += per_row * __popcll(there);
            level--;
            there = __ballot(tiles > level);
        }
        if (level < 0) return false;
        const int rank = (idx - base) / per_row;
        group = idx - base - rank * per_row;
        const uint64_t nth =
            __ballot(((there >> lane) & 1) && __popcll(there & ((1ull << lane) - 1)) == rank);
        seq = __ffsll((unsigned long long)nth) - 1;
        tile = level;
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
