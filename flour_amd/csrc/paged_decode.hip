// paged_decode.hip — kernel (2): paged decode attention on gfx950 matrix cores.
//
// Replaces paged_attention (src/backend/cpu.rs:57-112) for one new query per sequence
// (seq_q == 1, the decode step engine.rs:259-262), batched over sequences. The block list of
// Cache::kv_blocks (cache.rs:456-458, KvCache::gather_blocks cache.rs:83-96) arrives as a
// block table; query head h reads kv head h / n_rep (repeat_kv, cpu.rs:5-13); with seq_q == 1
// the causal mask of cpu.rs:88-95 admits every cached position, so only positions past the
// context length are masked.
//
// Work decomposition (stream-K at wave granularity): the K/V to read is the list of 32-token
// chunks of every (sequence, kv head) pair, laid end to end. One resident round of one-wave
// workgroups (3 per CU) each takes an equal contiguous range of that list, so every
// wave streams the same number of bytes whatever the spread of context lengths, and no wave
// pays a launch or a ramp-up twice. A pair wholly inside one range is finished by its wave; a
// pair cut by range ends leaves one partial (max, sum, acc) row per piece, and a small second
// kernel on the same stream merges those (log-sum-exp merge, as in the running update of
// cpu.rs:96-105). The kernel boundary orders partial writes before merge reads; an in-kernel
// "last workgroup merges" scheme would need an agent-scope release/acquire per workgroup,
// which on this multi-XCD part writes back and invalidates the XCD's L2 each time.
//
// Inside a piece (bf16/f16 pools, head_dim 128 or 64, block_size a multiple of 16; the
// figures below are for head_dim 128, and head_dim 64 halves every row: 8-byte lane loads, a
// 128-byte row per 16 lanes, 16 output dims per lane instead of 32):
//  * The wave walks its piece chunk by chunk. A chunk is two 16-token MFMA tiles, each one
//    4 KB (head, 16 slots) pool run of K and of V, read with buffer loads (per-pool resource,
//    loop-invariant lane offset, per-tile SGPR offset; non-temporal, whole rows per
//    instruction; K is turned into the MFMA layout through LDS); two register buffers
//    ping-pong so the next chunk's loads are in flight while one is computed, with the loop
//    peeled so that no load is conditional. Every query head of the kv head shares each K/V
//    load (GQA reuse: K/V leave HBM once).
//  * Scores S = K Q^T on v_mfma_f32_16x16x32 (M = 16 tokens, N = 16 query-head columns, the
//    n_rep real heads padded with zero rows): lane (g, c) = (lane/16, lane%16) holds head c's
//    scores for tokens 4g..4g+3 of each tile.
//  * Those registers, for the two tiles, are exactly the B operand of v_mfma_f32_16x16x32 for
//    O^T = V^T P^T (K = the 32 tokens), so P never leaves the lane. The V^T A operand is built
//    in-lane: each lane loads V rows 4g..4g+3, dims 8c..8c+7 (a wave reads 4 whole 256 B rows
//    per instruction) and v_perm_b32 packs, per output dim 8c+n, the four tokens' values. The
//    O^T accumulator holds, in lane (g, c), query head c at dims 32g..32g+31.
//  * P is split into hi + lo 16-bit parts (two MFMAs per product) so the P.V contraction keeps
//    ~16 mantissa bits of P; products are exact in fp32 and accumulate in fp32.
//  * fp32 pools (longer steps, decode_f32_split): the same stream over 16-token chunks of the same
//    bytes, on v_mfma_f32_16x16x4 in fp32 end to end. A wave instruction reads four 256 B row
//    segments; the score registers are the B operand as they stand (one product per token group
//    and 16 dims) and V registers the A operand, so only K goes through LDS. HBM-bound: 16 x
//    256-2,048 tokens of 32 / 8 heads of 128 (129 MB) 108 us on the vector kernel, 36.8 here.
//  * Online softmax in the exp2 domain: the only cross-lane step per chunk is the max over the
//    four row groups (two v_permlane*_swap exchanges); running sums stay lane-partial until
//    the end, and the accumulator is rescaled only when some lane's max moved.
#include <math.h>

#include <atomic>
#include <mutex>
#include <type_traits>

#include "flour_common.h"

namespace flour {

bool simt_supported(int dtype, int head_dim, const void* q, int64_t q_st, int64_t q_sh,
                    const void* k_pool, const void* v_pool);
int launch_attn_simt(int dtype, int out_dtype, void* out, int64_t o_st, int64_t o_sh,
                     const void* q, int64_t q_st, int64_t q_sh, const void* k_pool,
                     const void* v_pool, const int32_t* cu, const int32_t* kv_lens,
                     const int32_t* bt, int max_blocks, int num_seqs, int total_q, int num_heads,
                     int n_rep, int head_dim, int block_size, int64_t num_slots, int max_kv,
                     float scale, hipStream_t stream);
int launch_attn_generic(int dtype, int out_dtype, void* out, int64_t o_st, int64_t o_sh,
                        const void* q, int64_t q_st, int64_t q_sh, const void* k_pool,
                        const void* v_pool, const int32_t* cu, const int32_t* kv_lens,
                        const int32_t* bt, int max_blocks, int num_seqs, int total_q,
                        int num_heads, int n_rep, int head_dim, int block_size, int64_t num_slots,
                        int max_kv, float scale, hipStream_t stream);

static constexpr float LOG2E = 1.4426950408889634f;

// Tokens per step: two 16-token MFMA tiles of a 16-bit pool, one of an fp32 pool (the same bytes)
__host__ __device__ constexpr int dec_chunk(int elem_bytes) { return elem_bytes == 4 ? 16 : 32; }
static constexpr int DEC_SEG = 32;           // chunks per tile-slot refill (up to 64 tiles, one per lane)
static constexpr int DEC_MAX_BATCH = 4096;   // per-sequence chunk prefix sums live in LDS
// Three waves per CU. Each wave keeps one 32-token chunk in flight while it computes the
// previous one (16 KB at head_dim 128), so 768 waves hold ~12 MB of reads, about HBM's
// bandwidth-delay product; more waves only lengthen the queues and open more DRAM rows at once
// on the random 4 KB page runs (measured on the Llama-3-8B / 70B / Qwen2.5-0.5B decode batches:
// 3 per CU stream 0.3-1.5% faster than 4, which stream 3-7% faster than 8; counts that do not
// divide evenly over a CU's 4 SIMDs, 2.5, 3.5 and 5 per CU, are slower than their neighbours).
static constexpr int DEC_WAVES_PER_CU = 3;
// fp32 pools: the fp32 products of a chunk keep a SIMD's matrix core busy for ~2,050 cycles of
// every 16 KB, so every SIMD gets a wave (3 / 4 / 6 per CU: 163 / 149 / 142 us for 855 MB at 32 / 8
// heads of 128, 131 / 126 / 136 us for 806 MB at 8 heads of 64).
static constexpr int DEC_WAVES_PER_CU_F32 = 4;
static_assert(DEC_WAVES_PER_CU_F32 >= DEC_WAVES_PER_CU, "the workspace is sized for the larger");
// K is read like V, four whole 256 B rows per instruction with the non-temporal hint, and
// turned into the MFMA A-operand layout (row = lane % 16) through a per-wave LDS tile. Reading
// K directly in that layout takes a 64 B quarter of 16 rows per instruction, a pattern that
// streams at most ~6.0 TB/s from HBM against ~6.8 TB/s for whole rows (measured with the same
// 2048-wave, double-buffered access over random 4 KB runs).
// Bytes per K row in LDS: the row and 16 bytes, conflict-free 16-byte fragment reads of 16 rows.
__host__ __device__ constexpr int dec_kpitch(int d, int elem_bytes) { return d * elem_bytes + 16; }

struct DecodeWs {
    float* ml;  // [2 * num_waves][n_rep][2] (max, sum) in the exp2 domain
    float* o;   // [2 * num_waves][n_rep][D]
    int* pre;   // [batch + 1] chunk prefix sums, written by workgroup 0 for the merge kernel
    // row of q / out that batch entry b reads and writes: rows[b], or b when null (a mixed
    // continuous-batching step runs its one-row sequences, scattered among the packed rows of
    // longer ones, as one decode batch)
    const int32_t* rows;
    // Decode step of a batch with its KV write fused in (the kernel's FUSE instantiation): the
    // new K / V row of entry b and kv head g at k_new / v_new + b * new_st + g * new_sh
    // (elements), written to pool slot new_slots[b] (skipped outside [0, num_slots)) before the
    // attention reads it.
    const void* k_new;
    const void* v_new;
    int64_t new_st, new_sh;
    const int32_t* new_slots;
    int xcd_w;  // wave-range weight w (WaveRanges): even ranges 32 + w, odd 32 - w
};

static int g_wg_override = 0;  // tuning / test hook: number of waves (0 = one resident round)
// Wave-range weight w of WaveRanges (0 .. 16): even-indexed ranges (even XCDs) take w/32 more
// chunks than the mean, odd ones w/32 fewer (a tuning / test switch). Same-box sweep of w = 0 ..
// 4: 2 is best or even on every decode workload (Llama-3-8B batch 5,862 -> 5,989 GB/s, 70B
// batch 6,083 -> 6,231, head_dim-64 batch even).
static int g_xcd_weight = 2;

static int decode_workgroups(int dtype) {
    const int per_cu = dtype == FLOUR_DTYPE_F32 ? DEC_WAVES_PER_CU_F32 : DEC_WAVES_PER_CU;
    const int n = g_wg_override > 0 ? g_wg_override : device_cus() * per_cu;
    return n < 4096 ? n : 4096;
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

static size_t decode_ws_bytes(int nwg, int n_rep, int head_dim, int batch) {
    const size_t slots = 2 * (size_t)nwg;
    return align256(slots * n_rep * 2 * sizeof(float)) +
           align256(slots * n_rep * (size_t)head_dim * sizeof(float)) +
           align256(((size_t)batch + 1) * sizeof(int));
}

template <int CHUNK>
__device__ __forceinline__ int decode_chunks(int ctx, int max_ctx) {
    ctx = min(ctx, max_ctx);
    return ctx > 0 ? (ctx + CHUNK - 1) / CHUNK : 0;
}

// Wave ranges over the flattened chunk list. The dispatcher places workgroup i on XCD i % 8,
// and on this path the odd XCDs stream 6-9% slower than their even partners (per-workgroup
// clock stamps: every pair, three machines, both head shapes), so the launch would wait for the
// odd half. Even-indexed ranges therefore hold w/32 more chunks than the mean and odd ones w/32
// fewer: range i is [lo(i), lo(i + 1)) with lo(i) = floor(total (32 i + w (i & 1)) / W),
// W = 32 n + w (n & 1), so lo(0) = 0 and lo(n) = total. The split depends on the shapes alone,
// never on timing, so results stay deterministic. I is uint32_t when total * (W + 32) fits 32
// bits (a 64-bit division is a long instruction sequence), else int64_t.
template <typename I>
struct WaveRanges {
    I total, n, w, W;
    __device__ WaveRanges(int64_t total_, int64_t n_, int w_)
        : total((I)total_), n((I)n_), w((I)w_), W((I)(32 * n_ + w_ * (n_ & 1))) {}
    __device__ I lo(I i) const { return total * (32 * i + w * (i & 1)) / W; }
    // the range holding chunk x (0 <= x < total): the last i < n with lo(i) <= x (the estimate
    // is within a range or two of it, as no range differs from the mean by more than w/32)
    __device__ I owner(I x) const {
        I i = x * W / (32 * total);
        if (i > n - 1) i = n - 1;
        while (i + 1 < n && lo(i + 1) <= x) i++;
        while (i > 0 && lo(i) > x) i--;
        return i;
    }
};

// Whether every numerator of WaveRanges fits 32 bits: up to ~174,500 chunks on 768 waves (64 x 10.9K
// tokens over 8 kv heads of a 16-bit pool), ~131,000 on 1,024 (64 x 4.1K of an fp32 one).
__device__ __forceinline__ bool ranges_narrow(int64_t total, int64_t n, int w) {
    return (uint64_t)total * (uint64_t)(32 * n + w + 32) <= 0xffffffffull;
}

// Ranges that a list of `total` chunks is cut into by a grid of `cap` waves: at least two chunks
// each. Fewer, longer ranges leave fewer pieces to merge (one 2,000-token sequence of 8 kv heads,
// 504 chunks: 10.2 us on 252 waves, 10.9 on 504), a list of more than `cap` chunks has a range of
// two anyway, and no range is empty (the smallest share is (32 - w) / 32 >= 1/2 of the mean).
__device__ __forceinline__ int64_t range_count(int64_t total, int64_t cap) {
    const int64_t half = total >> 1;
    return half < 1 ? 1 : (half < cap ? half : cap);
}

// Running maxima start at the lowest finite value: with scores of -inf alone (K rows that hold -inf,
// products that overflow) the maximum stays finite, every weight is exp2(-inf) = 0 and no
// difference of infinities reaches the sums. It costs nothing where a select per chunk would.
static constexpr float DEC_M0 = -3.402823466e38f;

// What a row is divided by: its sum of weights, or 1 where that is 0 (no score above -inf: a zero
// row). Over fp32 pools an undefined sum (scores of NaN or +inf) gives a zero row too, as on the
// vector kernel (attn_simt.hip): the caller clears the row wherever !(sum > 0). The 16-bit pools
// hand a NaN on.
template <bool F32>
__device__ __forceinline__ float divisor(float sum) {
    return (F32 ? !(sum > 0.0f) : sum == 0.0f) ? 1.0f : sum;
}

__device__ __forceinline__ f32x4 mfma16x16x4_f32(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// One wave per workgroup; each wave owns one contiguous range of the chunk list. D is the head
// dim, 128 or 64. A lane's K/V share of a 16-token tile is rows 4lg .. 4lg + 3 at 16-byte
// (D 128: dims 8lc ..) or 8-byte (D 64: dims 4lc ..) width, so a wave reads whole rows.
template <typename T, typename TO, bool BS16, int D, bool FUSE>
__global__ __launch_bounds__(64, 2) void paged_decode_mfma_kernel(
    TO* __restrict__ out, const T* __restrict__ q, const T* __restrict__ k_pool,
    const T* __restrict__ v_pool, const int32_t* __restrict__ block_tables, int max_blocks,
    const int32_t* __restrict__ context_lens, int batch, int num_heads, int kv_heads, int n_rep,
    int block_size, int64_t num_slots, int max_ctx, float scale_log2, DecodeWs ws) {
    static_assert(D == 128 || D == 64, "matrix-core decode: head_dim 128 or 64");
    constexpr bool F32 = std::is_same<T, float>::value;
    constexpr int CHUNK = dec_chunk(sizeof(T));
    constexpr int TILES = CHUNK / 16;  // 16-token tiles per chunk
    constexpr int KP = dec_kpitch(D, sizeof(T));
    constexpr int NV = D / 16;  // O^T products per chunk (16 output dims each)
    // A lane's loads of K (and of V) per chunk: [NL][4] of Ld. 16-bit pools: tile t, row 4lg + j,
    // 8 (D 128) or 4 (D 64) dims. fp32 pools: row 4lg + j of the one tile, dims 64i + 4lc .. + 3,
    // so an instruction reads four 256-byte row segments in every form (128 at D 64, 16-bit).
    constexpr int NL = F32 ? D / 64 : TILES;
    typedef typename std::conditional<F32 || D == 128, u32x4, u32x2>::type Ld;
    extern __shared__ int pre[];  // pre[b] = chunks of sequences 0..b-1; pre[batch] = all
    __shared__ __attribute__((aligned(16))) unsigned char kt[16 * KP];  // one K tile
    const int lane = threadIdx.x, lg = lane >> 4, lc = lane & 15;

    // ---- exclusive prefix sum of per-sequence chunk counts. Up to 64 sequences stay in
    // registers, one per lane (clamped context length and prefix), so that locating a segment
    // is a ballot and scalar lane reads: no LDS search, no second read of a context length.
    // (16-token pages: with other page sizes those two registers spill)
    const bool in_lanes = BS16 && batch <= 64;
    int my_ctx = 0, my_pre = 0, all_chunks;
    if (in_lanes) {
        my_ctx = lane < batch ? min(context_lens[lane], max_ctx) : 0;
        const int n = decode_chunks<CHUNK>(my_ctx, max_ctx);
        const int incl = wave_incl_sum(n);
        my_pre = incl - n;
        all_chunks = __builtin_amdgcn_readlane(incl, 63);
        if constexpr (FUSE) {  // its walk over the pairs reads them by index
            if (lane < batch) pre[lane] = my_pre;
            if (lane == 63) pre[batch] = incl;
            __syncthreads();
        }
        if (blockIdx.x == 0) {  // for the merge kernel (ordered by the kernel boundary)
            if (lane < batch) ws.pre[lane] = my_pre;
            if (lane == 63) ws.pre[batch] = incl;
        }
    } else {  // each lane scans a slice, through LDS
        const int per = (batch + 63) / 64;
        int local = 0;
        for (int i = 0; i < per; i++) {
            const int b = lane * per + i;
            if (b < batch) local += decode_chunks<CHUNK>(context_lens[b], max_ctx);
        }
        const int incl = wave_incl_sum(local);
        int run = incl - local;
        for (int i = 0; i < per; i++) {
            const int b = lane * per + i;
            if (b < batch) {
                pre[b] = run;
                run += decode_chunks<CHUNK>(context_lens[b], max_ctx);
            }
        }
        if (lane == 63) pre[batch] = incl;
        __syncthreads();
        all_chunks = __builtin_amdgcn_readlane(incl, 63);
        if (blockIdx.x == 0)
            for (int b = lane; b <= batch; b += 64) ws.pre[b] = pre[b];
    }
    const int64_t total = (int64_t)kv_heads * all_chunks;
    const int64_t nwg = range_count(total, gridDim.x), wgi = blockIdx.x;
    if (total == 0 || wgi >= nwg) return;
    // 32-bit divisions whenever they fit: a 64-bit one is ~0.3 us of instructions, and the
    // range bounds and the first segments stand before the wave's first load
    const bool narrow = ranges_narrow(total, nwg, ws.xcd_w);
    // The range is [lo, lo + len); positions in it are 32-bit offsets from lo
    // (a range of 2^31 chunks would be 16 TB of reads). Everything that selects a segment is
    // uniform and made scalar here: a divergent value would put every
    // buffer load that takes its offset into a per-lane loop.
    int64_t lo;
    int len;
    if (narrow) {
        const WaveRanges<uint32_t> wr(total, nwg, ws.xcd_w);
        const uint32_t a = wr.lo((uint32_t)wgi);
        lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)a);
        len = __builtin_amdgcn_readfirstlane((int)(wr.lo((uint32_t)wgi + 1) - a));
    } else {
        const WaveRanges<int64_t> wr(total, nwg, ws.xcd_w);
        const int64_t a = wr.lo(wgi);
        lo = ((int64_t)__builtin_amdgcn_readfirstlane((int)(a >> 32)) << 32) |
             (uint32_t)__builtin_amdgcn_readfirstlane((int)a);
        len = __builtin_amdgcn_readfirstlane((int)(wr.lo(wgi + 1) - a));
    }

    const uint32_t head_bytes = (uint32_t)(num_slots * D * (int64_t)sizeof(T));
    // K and V: instruction j of a tile reads rows 4lg + j, dims (D / 16) lc .. (4 whole rows)
    uint32_t v_off = (uint32_t)((4 * lg * D + (F32 ? 4 : D / 16) * lc) * sizeof(T));
    // opaque: with its low bits known, the row offsets become ORs held in a register each instead
    // of the loads' immediate offsets
    asm volatile("" : "+v"(v_off));
    const int64_t max_phys = num_slots / block_size - 1;

    // The wave's range is a stream of segments: up to DEC_SEG consecutive chunks of one
    // (sequence, kv head) pair. Consecutive segments of the same pair form one piece.
    struct Seg {
        int b, g, cb, ce, nch, tok_end;
    };
    auto seg_at = [&](int at) -> Seg {
        const int64_t x = lo + at;
        Seg sg;
        int before, ctx;  // chunks per head before sequence b, its clamped context length
        if (in_lanes) {   // largest b with kv_heads * pre[b] <= x
            const uint64_t le = __ballot(lane < batch && (int64_t)kv_heads * my_pre <= x);
            sg.b = __popcll(le) - 1;
            before = __builtin_amdgcn_readlane(my_pre, sg.b);
            ctx = __builtin_amdgcn_readlane(my_ctx, sg.b);
            sg.nch = decode_chunks<CHUNK>(ctx, max_ctx);
        } else {
            int l0 = 0, h0 = batch;
            while (h0 - l0 > 1) {
                const int mid = (l0 + h0) >> 1;
                if ((int64_t)kv_heads * pre[mid] <= x)
                    l0 = mid;
                else
                    h0 = mid;
            }
            sg.b = __builtin_amdgcn_readfirstlane(l0);
            before = __builtin_amdgcn_readfirstlane(pre[l0]);
            sg.nch = __builtin_amdgcn_readfirstlane(pre[l0 + 1]) - before;
            ctx = min(context_lens[sg.b], max_ctx);
        }
        const int64_t rel = x - (int64_t)kv_heads * before;
        sg.g = __builtin_amdgcn_readfirstlane(narrow ? (int)((uint32_t)rel / (uint32_t)sg.nch)
                                                     : (int)(rel / sg.nch));
        sg.cb = (int)(rel - (int64_t)sg.g * sg.nch);
        sg.ce = sg.cb + min(min(sg.nch - sg.cb, DEC_SEG), len - at);
        sg.tok_end = min(ctx, sg.ce * CHUNK);
        return sg;
    };
    // Pool slot of the first token of each tile of a segment: lane i holds tile i (chunk
    // cb + i/2, half i%2), so the loop fetches it with v_readlane. Tiles past the segment are
    // clamped to its last tile: every address stays valid, their tokens are masked and their V
    // zeroed in compute_chunk.
    // The block id is kept as loaded and clamped only where a tile load reads it (one segment
    // later for the next segment): using it here would make the wave wait for this load, and
    // with it for every chunk load in flight.
    struct Slots {
        int id, off;  // lane i: block id and in-block offset of tile i's first token
    };
    const int max_id = (int)max_phys;
    auto seg_slots = [&](const Seg& sg) -> Slots {
        const int32_t* bt = block_tables + (int64_t)sg.b * max_blocks;
        const int last_tile_tok0 = ((sg.tok_end - 1) >> 4) << 4;
        const int tok0 = min(sg.cb * CHUNK + lane * 16, last_tile_tok0);
        const int lb = BS16 ? (tok0 >> 4) : tok0 / block_size;
        return Slots{bt[lb], BS16 ? 0 : tok0 - lb * block_size};
    };
    // Chunk loads as buffer loads: one resource per pool (the kv head's region), the
    // loop-invariant lane offset (VGPR) and the tile's byte offset (SGPR), so there is no
    // per-lane address arithmetic in the loop; non-temporal (K/V are read exactly once);
    // an out-of-region offset reads zeros instead of faulting.
    auto load_chunk = [&](int g, Slots sl, int tile0, Ld (*kd)[4], Ld (*vd)[4]) {
        const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(k_pool + (int64_t)g * num_slots * D), (short)0, (int)head_bytes, BUF_DWORD3);
        const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(v_pool + (int64_t)g * num_slots * D), (short)0, (int)head_bytes, BUF_DWORD3);
#pragma unroll
        for (int t = 0; t < TILES; t++) {
            int id = __builtin_amdgcn_readlane(sl.id, tile0 + t);
            id = id < 0 ? 0 : (id > max_id ? max_id : id);  // a bad block id never leaves the pool
            const uint32_t slot =
                BS16 ? (uint32_t)(id * 16)
                     : (uint32_t)(id * block_size + __builtin_amdgcn_readlane(sl.off, tile0 + t));
            const uint32_t soff = slot * (uint32_t)(D * sizeof(T));
            auto load_rows = [&](const __amdgpu_buffer_rsrc_t& rsrc, Ld (*d)[4]) {
#pragma unroll
                for (int i = 0; i < NL / TILES; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const uint32_t off = v_off + (j * D + 64 * i) * (uint32_t)sizeof(T);
                        if constexpr (sizeof(Ld) == 16)
                            d[t + i][j] =
                                __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, soff, BUF_NT);
                        else
                            d[t + i][j] =
                                __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, soff, BUF_NT);
                    }
            };
            load_rows(k_rsrc, kd);
            load_rows(v_rsrc, vd);
        }
    };
    // Q^T as the B operand: lane (lg, lc) holds head lc, dims 32kk + 8lg .. +7; fp32: dims
    // 16kk + 4lg .. + 3, one per k-step 4kk .. 4kk + 3.
    constexpr int NQ = D * (int)sizeof(T) / 64;
    u32x4 qb[NQ];
    auto load_q = [&](int b, int g) {
        const int64_t row = ws.rows ? (int64_t)ws.rows[b] : (int64_t)b;
        const T* qh = q + (row * num_heads + (int64_t)g * n_rep + lc) * D + (F32 ? 4 : 8) * lg;
#pragma unroll
        for (int kk = 0; kk < NQ; kk++)
            qb[kk] = (lc < n_rep) ? *reinterpret_cast<const u32x4*>(qh + (F32 ? 16 : 32) * kk)
                                  : u32x4{0, 0, 0, 0};
    };

    float m = DEC_M0, lsum = 0.0f;
    f32x4 acc[NV];
#pragma unroll
    for (int nn = 0; nn < NV; nn++) acc[nn] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto compute_chunk = [&](int c, int tok_end, Ld (*ka)[4], Ld (*va)[4]) {
        const int tok0 = c * CHUNK;
        const bool full = tok0 + CHUNK <= tok_end;
        if (!full) {  // tokens past the context: zero V so garbage bits cannot leak in
#pragma unroll
            for (int t = 0; t < NL; t++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (tok0 + (F32 ? 0 : 16 * t) + 4 * lg + j >= tok_end) va[t][j] = Ld{};
        }
        // K rows through LDS into the A-operand layout: lane (lg, lc) needs row lc, dims
        // 32kk + 8lg .. +7 (fp32: 16kk + 4lg .. + 3). One wave per workgroup and LDS operations
        // of a wave complete in order, so the wave barriers only keep the compiler from moving
        // LDS accesses across. The second tile's writes follow the first tile's reads in that
        // order.
        u32x4 kA[TILES][NQ];
#pragma unroll
        for (int t = 0; t < TILES; t++) {
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < NL / TILES; i++)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    *reinterpret_cast<Ld*>(&kt[(4 * lg + j) * KP + 256 * i + (int)sizeof(Ld) * lc]) =
                        ka[t + i][j];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int kk = 0; kk < NQ; kk++)
                kA[t][kk] = *reinterpret_cast<const u32x4*>(&kt[lc * KP + 64 * kk + 16 * lg]);
        }
        __builtin_amdgcn_wave_barrier();
        // S tiles: s[t][r] = score of head lc for token 16t + 4lg + r of the chunk.
        f32x4 s[TILES];
#pragma unroll
        for (int t = 0; t < TILES; t++) {
            s[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (F32) {
                // Sums of 8 products, added pairwise: one chain over the D products of a score has
                // ~1.3 times the vector kernel's rounding error on short contexts.
                f32x4 lvl[4];  // lvl[n]: a pending sum of 2^n k-steps
#pragma unroll
                for (int kk = 0; kk < NQ; kk++) {
                    f32x4 h[2] = {s[t], s[t]};
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        h[e >> 1] = mfma16x16x4_f32(__uint_as_float(kA[t][kk][e]),
                                                    __uint_as_float(qb[kk][e]), h[e >> 1]);
                    f32x4 x = h[0] + h[1];
                    int n = 0;
                    for (; (kk >> n) & 1; n++) x = lvl[n] + x;
                    lvl[n] = x;
                    if (kk & 1) __builtin_amdgcn_sched_barrier(0);  // (few pending sums)
                }
                s[t] = lvl[NQ == 8 ? 3 : 2];
                __builtin_amdgcn_sched_barrier(0);  // (registers: no V^T P^T before the scores)
            } else {
#pragma unroll
                for (int kk = 0; kk < NQ; kk++) s[t] = mfma16x16x32<T>(kA[t][kk], qb[kk], s[t]);
            }
        }
        float sv[4 * TILES];
        float tmax = -INFINITY;
#pragma unroll
        for (int t = 0; t < TILES; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const bool ok = full || (tok0 + 16 * t + 4 * lg + r < tok_end);
                sv[4 * t + r] = ok ? s[t][r] * scale_log2 : -INFINITY;
                tmax = fmaxf(tmax, sv[4 * t + r]);
            }
        tmax = max_across_rows(tmax);
        const float m_new = fmaxf(m, tmax);
        const float alpha = fast_exp2(m - m_new);
        float p[4 * TILES];
#pragma unroll
        for (int i = 0; i < 4 * TILES; i++)  // fp32: the scaling and the difference round once
            p[i] = fast_exp2(F32 ? (sv[i] == -INFINITY ? sv[i] : fmaf(s[0][i & 3], scale_log2, -m_new))
                                 : sv[i] - m_new);
        float psum = (p[0] + p[1]) + (p[2] + p[3]);
        if constexpr (TILES == 2) psum += (p[4] + p[5]) + (p[6] + p[7]);
        lsum = lsum * alpha + psum;
        if (__builtin_amdgcn_ballot_w64(m_new > m) != 0) {
#pragma unroll
            for (int nn = 0; nn < NV; nn++) acc[nn] *= alpha;
        }
        m = m_new;
        if constexpr (F32) {
            // O^T += V^T P^T, one product per score register j and 16-dim block nn = 4i + e: B is
            // the lane's p[j] (token 4lg + j, head lc), A the lane's V at that token, dim
            // 64i + 4lc + e. The chunk is summed by itself and then added, so a long context's sum
            // is a sum of chunk sums (fp32 rounding: relative error against 64 bits of 16 x 256-
            // 2,048 tokens 2.7e-7 with one chain, the vector kernel 2.0e-7).
#pragma unroll
            for (int nn = 0; nn < NV; nn++) {
                f32x4 t = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int j = 0; j < 4; j++)
                    t = mfma16x16x4_f32(__uint_as_float(va[nn >> 2][j][nn & 3]), p[j], t);
                acc[nn] += t;
            }
        } else {
            // P^T as the B operand over the 32 tokens: lane (lg, lc) holds head lc at
            // k-slots 8lg + j: j < 4 -> token 4lg + j (tile 0), j >= 4 -> 16 + 4lg + j - 4.
            // Split hi + lo so the product keeps ~16 mantissa bits of P.
            u32x4 PH, PL;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint32_t hi16 = pack2<T>(p[2 * i], p[2 * i + 1]);
                PH[i] = hi16;
                PL[i] = pack2<T>(p[2 * i] - lo_f32<T>(hi16), p[2 * i + 1] - hi_f32<T>(hi16));
            }
            // V^T as the A operand: lane (lg, lc) holds output dim (D / 16) lc + nn at the same
            // k-slots, packed in-lane from its four V rows of each tile.
#pragma unroll
            for (int nn = 0; nn < NV; nn++) {
                const int wd = nn >> 1;
                u32x4 A;
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    if (nn & 1) {
                        A[2 * t] = perm_hi16(va[t][0][wd], va[t][1][wd]);
                        A[2 * t + 1] = perm_hi16(va[t][2][wd], va[t][3][wd]);
                    } else {
                        A[2 * t] = perm_lo16(va[t][0][wd], va[t][1][wd]);
                        A[2 * t + 1] = perm_lo16(va[t][2][wd], va[t][3][wd]);
                    }
                }
                acc[nn] = mfma16x16x32<T>(A, PH, acc[nn]);
                acc[nn] = mfma16x16x32<T>(A, PL, acc[nn]);
            }
        }
    };

    // Piece epilogue from registers: lane (lg, lc) holds head lc, dims (D / 4) lg + NV r + nn
    // (r < 4, nn < NV): D / 4 contiguous dims; fp32 pools: dims 64i + 16lg + 4r + e for nn = 4i + e.
    auto epilogue = [&](int b, int g, bool complete, bool first_piece) {
        lsum = sum_across_rows(lsum);
        // lg made opaque here, so the per-lane output addresses are formed at the store instead
        // of being hoisted out of the stream as 64-bit values (which spill, and a spill reload
        // waits for every chunk load in flight)
        int lgo = lg;
        asm volatile("" : "+v"(lgo));
        if (lc < n_rep) {
            if (complete) {  // whole pair in this range: final output
                const int64_t row = ws.rows ? (int64_t)ws.rows[b] : (int64_t)b;
                TO* o = out + (row * num_heads + (int64_t)g * n_rep + lc) * D +
                        (F32 ? 16 : D / 4) * lgo;
                const float inv = 1.0f / divisor<F32>(lsum);
                if (F32 && !(lsum > 0.0f))
#pragma unroll
                    for (int nn = 0; nn < NV; nn++) acc[nn] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if constexpr (F32) {
#pragma unroll
                        for (int h4 = 0; h4 < NV; h4 += 4) {
                            const f32x4 v = f32x4{acc[h4][r] * inv, acc[h4 + 1][r] * inv,
                                                  acc[h4 + 2][r] * inv, acc[h4 + 3][r] * inv};
                            if constexpr (sizeof(TO) == 4)
                                *reinterpret_cast<f32x4*>(o + 16 * h4 + 4 * r) = v;
                            else
                                *reinterpret_cast<u32x2*>(o + 16 * h4 + 4 * r) =
                                    u32x2{pack2<TO>(v[0], v[1]), pack2<TO>(v[2], v[3])};
                        }
                    } else if constexpr (sizeof(TO) == 4) {
#pragma unroll
                        for (int h4 = 0; h4 < NV; h4 += 4)
                            *reinterpret_cast<f32x4*>(o + NV * r + h4) =
                                f32x4{acc[h4][r] * inv, acc[h4 + 1][r] * inv, acc[h4 + 2][r] * inv,
                                      acc[h4 + 3][r] * inv};
                    } else {
                        uint32_t v[NV / 2];
#pragma unroll
                        for (int i = 0; i < NV / 2; i++)
                            v[i] = pack2<TO>(acc[2 * i][r] * inv, acc[2 * i + 1][r] * inv);
                        if constexpr (NV == 8)
                            *reinterpret_cast<u32x4*>(o + NV * r) = u32x4{v[0], v[1], v[2], v[3]};
                        else
                            *reinterpret_cast<u32x2*>(o + NV * r) = u32x2{v[0], v[1]};
                    }
                }
            } else {  // partial row for the merge kernel
                const int64_t pidx = (2 * wgi + (first_piece ? 0 : 1)) * n_rep + lc;
                float* o = ws.o + pidx * D + (F32 ? 16 : D / 4) * lgo;
#pragma unroll
                for (int r = 0; r < 4; r++)
#pragma unroll
                    for (int h4 = 0; h4 < NV; h4 += 4)
                        *reinterpret_cast<f32x4*>(o + (F32 ? 16 * h4 + 4 * r : NV * r + h4)) =
                            f32x4{acc[h4][r], acc[h4 + 1][r], acc[h4 + 2][r], acc[h4 + 3][r]};
                if (lg == 0) {
                    ws.ml[2 * pidx] = m;
                    ws.ml[2 * pidx + 1] = lsum;
                }
            }
        }
        m = DEC_M0;
        lsum = 0.0f;
#pragma unroll
        for (int nn = 0; nn < NV; nn++) acc[nn] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    };

    // ---- the chunk stream. The next segment's block-table slots are read while the current
    // one streams, and the two register buffers ping-pong across segment and piece boundaries:
    // the next chunk's loads (chosen with uniform selects, never a branch, so the compiler's
    // wait counts stay exact) are in flight while the current chunk is computed and while a
    // finished piece is written out.
    // FUSE: the new K / V row of every pair whose last chunk lies in this wave's range, written
    // to the pool before the range's first chunk load. The lanes that write a row, (lg, lc) with
    // 4 lg <= slot % 16 < 4 lg + 4 (the row's place in its 16-token tile, as the block table
    // places position context_len - 1), are the lanes that load it back in load_chunk, at the
    // same bytes (dims (D / 16) lc ..), so the wave's own program order makes the later load see
    // the row. No other wave reads the slot: the pair's last chunk, the only one holding the
    // new position, is in this range alone, and a batch's new slots are private to their
    // sequences. The first two pairs' rows are requested before the block-table and q loads
    // (their wait then overlaps those loads), stored after them; further pairs (short contexts)
    // two at a time after that.
    struct NewRows {
        int b, g, slot[2], pb[2], pg[2];
        bool pv[2], more;
        int first, nch;
        Ld kr[2], vr[2];
    };
    auto new_rows_load = [&](NewRows& nr) {
#pragma unroll
        for (int i = 0; i < 2; i++) {
            nr.pv[i] = nr.more;
            nr.pb[i] = nr.b;
            nr.pg[i] = nr.g;
            if (nr.more) {  // on to the next pair in the flattened order (sequences with chunks)
                nr.first += nr.nch;
                if (++nr.g == kv_heads) {
                    nr.g = 0;
                    do {
                        nr.b++;
                    } while (nr.b < batch && pre[nr.b + 1] == pre[nr.b]);
                }
                if (nr.b < batch) {
                    nr.nch = pre[nr.b + 1] - pre[nr.b];
                    nr.more = nr.first + nr.nch - 1 < len;
                } else {
                    nr.more = false;
                }
            }
        }
        const T* kn = static_cast<const T*>(ws.k_new);
        const T* vn = static_cast<const T*>(ws.v_new);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            nr.slot[i] = nr.pv[i] ? ws.new_slots[nr.pb[i]] : -1;
            if (nr.pv[i]) {
                const int64_t src = (int64_t)nr.pb[i] * ws.new_st + (int64_t)nr.pg[i] * ws.new_sh +
                                    (D / 16) * lc;
                nr.kr[i] = *reinterpret_cast<const Ld*>(kn + src);
                nr.vr[i] = *reinterpret_cast<const Ld*>(vn + src);
            }
        }
    };
    auto new_rows_store = [&](const NewRows& nr) {
        T* const kpw = const_cast<T*>(k_pool);
        T* const vpw = const_cast<T*>(v_pool);
#pragma unroll
        for (int i = 0; i < 2; i++) {
            const int sl = nr.slot[i];
            if (nr.pv[i] && sl >= 0 && sl < num_slots && lg == ((sl & 15) >> 2)) {
                const int64_t dst = ((int64_t)nr.pg[i] * num_slots + sl) * D + (D / 16) * lc;
                *reinterpret_cast<Ld*>(kpw + dst) = nr.kr[i];
                *reinterpret_cast<Ld*>(vpw + dst) = nr.vr[i];
            }
        }
    };

    Seg cur = seg_at(0);
    NewRows nr{};
    if constexpr (FUSE) {
        nr.b = cur.b;
        nr.g = cur.g;
        nr.nch = cur.nch;
        nr.first = -cur.cb;  // pair (b, g)'s first chunk, as an offset from lo
        nr.more = nr.first + nr.nch - 1 < len;
        new_rows_load(nr);
    }
    Slots cur_slots = seg_slots(cur);
    int nx = cur.ce - cur.cb;
    bool has_nxt = nx < len;
    Seg nxt = cur;
    Slots nxt_slots{0, 0};  // (not a copy of cur_slots, which would wait for its load)
    if (has_nxt) {
        nxt = seg_at(nx);
        nxt_slots = seg_slots(nxt);
    }
    int pc0 = cur.cb;  // first chunk of the current piece
    bool first_piece = true;
    int c = cur.cb;
    load_q(cur.b, cur.g);

    // One stream step: prefetch the chunk after c into (kn, vn) (PREFETCH is a compile-time
    // constant at each call, so the steady-state loop has no conditional loads), compute c
    // from (kc, vc), then advance the cursor.
    auto step = [&](auto prefetch, Ld (*kc)[4], Ld (*vc)[4], Ld (*kn)[4], Ld (*vn)[4]) {
        const bool seg_end = c + 1 >= cur.ce;
        // At a segment's last chunk the segment after the next one is looked up and its
        // block-table entries are requested before this step's chunk loads, so the rotation at
        // the end of the step waits for that load alone and not for the chunk loads behind it.
        int nn_x = nx;
        bool has_nn = false;
        Seg nn = nxt;
        Slots nn_slots = nxt_slots;
        if (seg_end && has_nxt) {
            nn_x = nx + (nxt.ce - nxt.cb);
            has_nn = nn_x < len;
            if (has_nn) {
                nn = seg_at(nn_x);
                nn_slots = seg_slots(nn);
            }
        }
        if constexpr (decltype(prefetch)::value) {
            const bool in_cur = c + 1 < cur.ce;
            const int pg = in_cur ? cur.g : nxt.g;
            const Slots pslots = in_cur ? cur_slots : nxt_slots;
            const int ptile = in_cur ? TILES * (c + 1 - cur.cb) : 0;
            load_chunk(pg, pslots, ptile, kn, vn);
        }
        compute_chunk(c, cur.tok_end, kc, vc);
        if (!seg_end) {
            c += 1;
            return;
        }
        // end of a segment
        const bool piece_end = !has_nxt || nxt.b != cur.b || nxt.g != cur.g;
        if (piece_end) epilogue(cur.b, cur.g, pc0 == 0 && cur.ce == cur.nch, first_piece);
        if (!has_nxt) return;
        if (piece_end) {
            pc0 = nxt.cb;
            first_piece = false;
            load_q(nxt.b, nxt.g);
        }
        cur = nxt;
        cur_slots = nxt_slots;
        c = cur.cb;
        nx = nn_x;
        has_nxt = has_nn;
        if (has_nn) {
            nxt = nn;
            nxt_slots = nn_slots;
        }
    };


    if constexpr (FUSE) {
        new_rows_store(nr);
        while (nr.more) {
            new_rows_load(nr);
            new_rows_store(nr);
        }
        asm volatile("" ::: "memory");  // the stores stay before the chunk loads
    }

    using pf_on = std::integral_constant<bool, true>;
    using pf_off = std::integral_constant<bool, false>;
    Ld ka[NL][4], va[NL][4], kb[NL][4], vb[NL][4];
    load_chunk(cur.g, cur_slots, 0, ka, va);
    int remaining = len;  // chunks this wave computes; all but the last prefetch one
    for (; remaining > 2; remaining -= 2) {
        step(pf_on{}, ka, va, kb, vb);
        step(pf_on{}, kb, vb, ka, va);
    }
    if (remaining == 2) {
        step(pf_on{}, ka, va, kb, vb);
        step(pf_off{}, kb, vb, ka, va);
    } else {
        step(pf_off{}, ka, va, kb, vb);
    }
}

// Merge of the pieces of pairs cut by wave ranges, and zero rows for empty contexts: one
// workgroup per (query head, sequence), lane i owning output dims 2i and 2i + 1, locating its
// pieces from the chunk prefix sums the main kernel left in the workspace. Pieces are taken 64 at
// a time (one per lane): their (max, sum) pairs become weights through wave reductions, then every
// lane accumulates its two dims over the batch with independent loads, reading each piece's
// weight and slot from the lane that holds it; batches combine with the same online rescaling
// as the running update of cpu.rs:96-105. With many pieces per pair (few sequences) the
// workgroup's waves split them, since one wave reads them 8 rows a memory round trip, and fold
// their states through LDS; with one wave there is no LDS and no barrier.
static constexpr int DEC_MERGE_WAVES = 8;
template <typename TO, int D, bool F32>
__global__ __launch_bounds__(64 * DEC_MERGE_WAVES) void paged_decode_merge_kernel(
    TO* __restrict__ out, int batch, int num_heads, int kv_heads, int n_rep, int nwg_i,
    DecodeWs ws) {
    // lane i owns output dims E i .. E i + E - 1
    constexpr int E = D / 64;
    const int h = blockIdx.x, b = blockIdx.y, lane = threadIdx.x & 63;
    const int w_id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    // chunks before sequence b, of sequence b and in all sequences (the main kernel's sums)
    const int before = ws.pre[b], nch = ws.pre[b + 1] - before, all = ws.pre[batch];
    const int64_t orow = ws.rows ? (int64_t)ws.rows[b] : (int64_t)b;
    TO* o = out + (orow * num_heads + h) * D + E * lane;
    if (nch == 0) {
        if (w_id == 0)
#pragma unroll
            for (int i = 0; i < E; i++) o[i] = from_f32<TO>(0.0f);
        return;
    }
    const int g = h / n_rep, hh = h - g * n_rep;
    const int64_t total = (int64_t)kv_heads * all, nwg = range_count(total, nwg_i);
    const int64_t s = (int64_t)kv_heads * before + (int64_t)g * nch;
    const int64_t e = s + nch;
    const bool narrow = ranges_narrow(total, nwg, ws.xcd_w);
    const WaveRanges<uint32_t> r32(narrow ? total : 1, nwg, ws.xcd_w);
    const WaveRanges<int64_t> r64(total, nwg, ws.xcd_w);
    auto range_lo = [&](int64_t i) -> int64_t {
        return narrow ? (int64_t)r32.lo((uint32_t)i) : r64.lo(i);
    };
    const int64_t f = narrow ? (int64_t)r32.owner((uint32_t)s) : r64.owner(s);
    const int64_t l = narrow ? (int64_t)r32.owner((uint32_t)(e - 1)) : r64.owner(e - 1);
    const bool f_first = s == range_lo(f);
    if (f == l) return;  // finished inside one wave range
    const int np = (int)(l - f + 1);  // ranges f..l, none of them empty

    float M = DEC_M0, L = 0.0f, O[E];
#pragma unroll
    for (int i = 0; i < E; i++) O[i] = 0.0f;
    const int fslot = (int)(f_first ? 2 * f : 2 * f + 1);  // the first piece always exists
    auto piece_slot = [&](int64_t p) -> int {  // slot of piece p (< np)
        const int64_t ij = f + p;
        return (int)((ij == f && !f_first) ? 2 * ij + 1 : 2 * ij);
    };
    typedef typename std::conditional<E == 2, f32x2, float>::type RowV;
    auto row = [&](int slot) -> RowV {  // this lane's E dims of a piece's partial row
        return *reinterpret_cast<const RowV*>(ws.o + ((int64_t)slot * n_rep + hh) * D + E * lane);
    };
    auto add = [&](float wj, RowV v) {
        if constexpr (E == 2) {
            O[0] += wj * v[0];
            O[1] += wj * v[1];
        } else {
            O[0] += wj * v;
        }
    };
    // this wave's pieces: an equal share
    const int per = waves == 1 ? np : (np + waves - 1) / waves;
    const int p_end = min(np, (w_id + 1) * per);
    for (int p0 = w_id * per; p0 < p_end; p0 += 64) {
        // The batch's first 8 pieces' rows are loaded before the (max, sum) reductions, which
        // they do not depend on (a missing piece reads the first piece's row, weight 0).
        const int slot = p0 + lane < p_end ? piece_slot(p0 + lane) : -1;
        RowV v0[8];
        int s0[8];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            s0[j] = p0 + j < p_end ? piece_slot(p0 + j) : -1;
            v0[j] = row(s0[j] >= 0 ? s0[j] : fslot);
        }
        float mx = -INFINITY, lx = 0.0f;
        if (slot >= 0) {
            mx = ws.ml[2 * ((int64_t)slot * n_rep + hh)];
            lx = ws.ml[2 * ((int64_t)slot * n_rep + hh) + 1];
        }
        const float m_new = fmaxf(M, wave_max(mx));
        const float w = (slot >= 0) ? fast_exp2(mx - m_new) : 0.0f;
        const float bl = wave_sum(w * lx);
        const float c_old = fast_exp2(M - m_new);
        L = L * c_old + bl;
#pragma unroll
        for (int i = 0; i < E; i++) O[i] *= c_old;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float wj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), j));
            if (s0[j] >= 0) add(wj, v0[j]);
        }
        // The rest in groups of 8 unconditional loads (a missing piece reads the first piece's
        // row) so they are all in flight together; the select drops them, so stale workspace
        // bits (even NaN) never reach the sum.
        const int nb = min(64, p_end - p0);
        for (int q = 8; q < nb; q += 8) {
            RowV v[8];
            int sl[8];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                sl[j] = __builtin_amdgcn_readlane(slot, q + j);
                v[j] = row(sl[j] >= 0 ? sl[j] : fslot);
            }
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float wj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), q + j));
                if (sl[j] >= 0) add(wj, v[j]);
            }
        }
        M = m_new;
    }
    if (waves > 1) {  // the waves' states, folded by the first (it always has pieces)
        __shared__ float wM[DEC_MERGE_WAVES], wL[DEC_MERGE_WAVES];
        __shared__ float wO[DEC_MERGE_WAVES][E][64];
        if (lane == 0) {
            wM[w_id] = M;
            wL[w_id] = L;
        }
#pragma unroll
        for (int i = 0; i < E; i++) wO[w_id][i][lane] = O[i];
        __syncthreads();
        if (w_id != 0) return;
        // all states are read together; slots past the last wave with pieces read its own
        float mx[DEC_MERGE_WAVES], lx[DEC_MERGE_WAVES], ox[DEC_MERGE_WAVES][E];
        float Mt = M;
#pragma unroll
        for (int x = 1; x < DEC_MERGE_WAVES; x++) {
            const bool on = x < waves && x * per < np;
            const int y = on ? x : 0;
            mx[x] = on ? wM[y] : -INFINITY;
            lx[x] = wL[y];
#pragma unroll
            for (int i = 0; i < E; i++) ox[x][i] = wO[y][i][lane];
        }
#pragma unroll
        for (int x = 1; x < DEC_MERGE_WAVES; x++) Mt = fmaxf(Mt, mx[x]);
        const float f0 = fast_exp2(M - Mt);
        L *= f0;
#pragma unroll
        for (int i = 0; i < E; i++) O[i] *= f0;
#pragma unroll
        for (int x = 1; x < DEC_MERGE_WAVES; x++) {
            if (x < waves && x * per < np) {
                const float f = fast_exp2(mx[x] - Mt);
                L += lx[x] * f;
#pragma unroll
                for (int i = 0; i < E; i++) O[i] += ox[x][i] * f;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < E; i++) {
        const float x = O[i] / divisor<F32>(L);
        o[i] = from_f32<TO>(F32 && !(L > 0.0f) ? 0.0f : x);
    }
}

// Waves per merge workgroup: about eight pieces (one memory round trip) each, for twice the mean
// number of pieces per pair (longer contexts than the mean have more).
static int decode_merge_waves(int grid, int batch, int kv_heads) {
    const int64_t pieces = 2 * (int64_t)grid / ((int64_t)batch * kv_heads);
    int waves = 1;
    while (waves < DEC_MERGE_WAVES && 8 * waves < pieces) waves *= 2;
    return waves;
}

template <typename T, typename TO, int D>
static int launch_decode_mfma_d(void* out, const void* q, const void* k_pool, const void* v_pool,
                                const int32_t* bt, int max_blocks, const int32_t* ctx_lens,
                                int batch, int num_heads, int kv_heads, int n_rep, int block_size,
                                int64_t num_slots, int max_ctx, float scale, int nwg, DecodeWs ws,
                                hipStream_t stream) {
    const size_t lds = (size_t)(batch + 1) * sizeof(int);
    const bool fuse = ws.k_new != nullptr;
    if (fuse && (block_size != 16 || std::is_same<T, float>::value)) {
        set_error("paged_decode: the fused KV write needs 16-token pages of a 16-bit pool");
        return FLOUR_ERR_UNSUPPORTED;
    }
    auto kern = block_size == 16 ? paged_decode_mfma_kernel<T, TO, true, D, false>
                                 : paged_decode_mfma_kernel<T, TO, false, D, false>;
    if constexpr (!std::is_same<T, float>::value)
        if (fuse) kern = paged_decode_mfma_kernel<T, TO, true, D, true>;
    // no more waves than ranges (range_count) for contexts of max_ctx
    const int64_t chunk = dec_chunk(sizeof(T));
    const int64_t half = (int64_t)batch * kv_heads * ((max_ctx + chunk - 1) / chunk) / 2;
    const int grid = (int)(half < 1 ? 1 : half < nwg ? half : nwg);
    kern<<<dim3(grid), dim3(64), lds, stream>>>(
        static_cast<TO*>(out), static_cast<const T*>(q), static_cast<const T*>(k_pool),
        static_cast<const T*>(v_pool), bt, max_blocks, ctx_lens, batch, num_heads, kv_heads, n_rep,
        block_size, num_slots, max_ctx, scale * LOG2E, ws);
    int rc = check_hip(hipGetLastError(), "paged_decode launch");
    if (rc != FLOUR_OK) return rc;
    const int mw = decode_merge_waves(grid, batch, kv_heads);
    paged_decode_merge_kernel<TO, D, std::is_same<T, float>::value>
        <<<dim3(num_heads, batch), dim3(64 * mw), 0, stream>>>(
            static_cast<TO*>(out), batch, num_heads, kv_heads, n_rep, grid, ws);
    return check_hip(hipGetLastError(), "paged_decode merge launch");
}

template <typename T, typename TO>
static int launch_decode_mfma(int head_dim, void* out, const void* q, const void* k_pool,
                              const void* v_pool, const int32_t* bt, int max_blocks,
                              const int32_t* ctx_lens, int batch, int num_heads, int kv_heads,
                              int n_rep, int block_size, int64_t num_slots, int max_ctx,
                              float scale, int nwg, DecodeWs ws, hipStream_t stream) {
    if (head_dim == 64)
        return launch_decode_mfma_d<T, TO, 64>(out, q, k_pool, v_pool, bt, max_blocks, ctx_lens,
                                               batch, num_heads, kv_heads, n_rep, block_size,
                                               num_slots, max_ctx, scale, nwg, ws, stream);
    return launch_decode_mfma_d<T, TO, 128>(out, q, k_pool, v_pool, bt, max_blocks, ctx_lens,
                                            batch, num_heads, kv_heads, n_rep, block_size,
                                            num_slots, max_ctx, scale, nwg, ws, stream);
}

}  // namespace flour

using namespace flour;

namespace flour {
__global__ void empty_kernel() {}
}  // namespace flour

// One empty one-wave workgroup on `stream`: the floor of a kernel launch on this device, timed
// beside the smallest decode workloads (a measurement helper, not part of the header).
extern "C" int flour_hip_empty_launch(void* stream) {
    flour::empty_kernel<<<dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream)>>>();
    return check_hip(hipGetLastError(), "empty launch");
}

extern "C" int flour_hip_set_decode_xcd_weight(int w) {
    if (w < 0 || w > 16) return FLOUR_ERR_INVALID_ARGUMENT;
    g_xcd_weight = w;
    return FLOUR_OK;
}

extern "C" int flour_hip_set_decode_workgroups(int n) {
    if (n < 0 || n > 4096) return FLOUR_ERR_INVALID_ARGUMENT;
    g_wg_override = n;
    return FLOUR_OK;
}

extern "C" int flour_hip_paged_decode_workspace_size(int batch, int num_heads, int kv_heads,
                                                     int head_dim, int max_context_len,
                                                     size_t* bytes) {
    clear_error();
    if (!bytes || batch < 0 || num_heads <= 0 || kv_heads <= 0 || num_heads % kv_heads != 0 ||
        head_dim <= 0 || max_context_len < 0) {
        set_error("paged_decode_workspace_size: bad arguments");
        return FLOUR_ERR_INVALID_ARGUMENT;
    }
    *bytes = decode_ws_bytes(decode_workgroups(FLOUR_DTYPE_F32), num_heads / kv_heads, head_dim, batch);
    return FLOUR_OK;
}

namespace flour {

// Body of flour_hip_paged_decode. `workspace` == nullptr with `ws_from_scratch` set takes the
// split-context workspace from this device's copy of `scratch` (flour_hip_paged_decode_noalloc).
static int paged_decode_impl(void* out, int out_dtype, const void* q, const void* k_pool,
                             const void* v_pool, const int32_t* block_tables,
                             int max_blocks_per_seq, const int32_t* context_lens, int batch,
                             int num_heads, int kv_heads, int head_dim, int block_size,
                             int64_t num_slots, int max_context_len, float scale, int dtype,
                             void* workspace, size_t workspace_bytes, bool ws_from_scratch,
                             const int32_t* rows, const DecodeWs* fused, void* stream);

// ------------------------------------------------------------------ allocation-free variant
// The split-context workspace of flour_hip_paged_decode_noalloc lives in this file-scope device
// array: each device the library runs on holds its own copy, for the life of the process. Host
// code never passes the array's name to a kernel or a copy (on the host it is a stand-in, not a
// device address): it uses the per-device address that hipGetSymbolAddress returns, looked up
// once per device on that device's first call.
static constexpr size_t DEC_SCRATCH_BYTES = (size_t)40 << 20;
static __device__ __align__(256) unsigned char scratch[DEC_SCRATCH_BYTES];
static constexpr int DEC_MAX_DEVICES = 64;
static std::atomic<void*> g_scratch_ptr[DEC_MAX_DEVICES];
static std::mutex g_scratch_mu;

static int scratch_for_current_device(void** ptr) {
    int dev = -1;
    const hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return check_hip(e, "paged_decode_noalloc: hipGetDevice");
    if (dev < 0 || dev >= DEC_MAX_DEVICES) {
        set_error("paged_decode_noalloc: device %d out of range", dev);
        return FLOUR_ERR_UNSUPPORTED;
    }
    void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
        if (!p) {
            const hipError_t r = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
            if (r != hipSuccess || !p)
                return check_hip(r != hipSuccess ? r : hipErrorInvalidSymbol,
                                 "paged_decode_noalloc: hipGetSymbolAddress(scratch)");
            g_scratch_ptr[dev].store(p, std::memory_order_release);
        }
    }
    *ptr = p;
    return FLOUR_OK;
}

}  // namespace flour

extern "C" int flour_hip_paged_decode(void* out, int out_dtype, const void* q,
                                      const void* k_pool, const void* v_pool,
                                      const int32_t* block_tables, int max_blocks_per_seq,
                                      const int32_t* context_lens, int batch, int num_heads,
                                      int kv_heads, int head_dim, int block_size,
                                      int64_t num_slots, int max_context_len, float scale,
                                      int dtype, void* workspace, size_t workspace_bytes,
                                      void* stream) {
    clear_error();
    return flour::paged_decode_impl(out, out_dtype, q, k_pool, v_pool, block_tables,
                                    max_blocks_per_seq, context_lens, batch, num_heads, kv_heads,
                                    head_dim, block_size, num_slots, max_context_len, scale, dtype,
                                    workspace, workspace_bytes, false, nullptr, nullptr, stream);
}

extern "C" size_t flour_hip_paged_decode_noalloc_max_workspace(void) {
    return flour::DEC_SCRATCH_BYTES;
}

extern "C" int flour_hip_paged_decode_noalloc(void* out, int out_dtype, const void* q,
                                              const void* k_pool, const void* v_pool,
                                              const int32_t* block_tables,
                                              int max_blocks_per_seq,
                                              const int32_t* context_lens, int batch,
                                              int num_heads, int kv_heads, int head_dim,
                                              int block_size, int64_t num_slots,
                                              int max_context_len, float scale, int dtype,
                                              void* stream) {
    clear_error();
    return flour::paged_decode_impl(out, out_dtype, q, k_pool, v_pool, block_tables,
                                    max_blocks_per_seq, context_lens, batch, num_heads, kv_heads,
                                    head_dim, block_size, num_slots, max_context_len, scale, dtype,
                                    nullptr, 0, true, nullptr, nullptr, stream);
}

namespace flour {

bool decode_mfma_supported(int dtype, int head_dim, int block_size, int n_rep, int batch,
                           int num_heads, int64_t num_slots, const void* q, const void* k_pool,
                           const void* v_pool) {
    return (dtype == FLOUR_DTYPE_BF16 || dtype == FLOUR_DTYPE_F16) &&
           (head_dim == 128 || head_dim == 64) && block_size % 16 == 0 && n_rep <= 16 &&
           batch <= DEC_MAX_BATCH && num_heads <= 65535 &&
           num_slots * head_dim * 2 <= (int64_t)0x7fffffff && ((uintptr_t)q % 16 == 0) &&
           ((uintptr_t)k_pool % 16 == 0) && ((uintptr_t)v_pool % 16 == 0);
}

// Whether an fp32 batch runs split over the chip on the matrix cores (with this workspace) rather
// than on the vector kernel, which needs no workspace but gives each (sequence, kv head) one
// workgroup.
static bool decode_f32_split(int head_dim, int block_size, int n_rep, int batch, int num_heads,
                             int64_t num_slots, int max_context_len, const void* out,
                             const void* q, const void* k_pool, const void* v_pool, bool ws_ok) {
    if (!ws_ok || (head_dim != 128 && head_dim != 64) || block_size % 16 != 0 || n_rep > 16 ||
        batch > DEC_MAX_BATCH || num_heads > 65535 ||
        num_slots * head_dim * 4 > (int64_t)0x7fffffff ||
        (((uintptr_t)out | (uintptr_t)q | (uintptr_t)k_pool | (uintptr_t)v_pool) & 15) != 0)
        return false;  // (its output stores are up to 16 bytes wide, the vector kernel's one element)
    // The vector kernel's time goes with a workgroup's kv length x queries (n_rep, as a power of
    // two) x head_dim; a split step takes ~9 us and its bytes. Vector / split in us: 1 x 256 tokens of
    // 32 / 8 heads of 128 14.5 / 10.3 (64 tokens: 7.4 / 9.8), 14 / 2 heads of 64 13.4 / 8.8 (64: 8.3 /
    // 8.4), 16 / 16 of 128 at 1,024 18.3 / 11.8 (256: 7.7 / 10.2), 8 / 8 of 64 at 2,048 19.9 / 10.0
    // (512: 8.1 / 9.0).
    int64_t work = (int64_t)max_context_len * head_dim, least = 131072;
    int nq = 1;
    for (; nq < n_rep && nq < 8; nq *= 2) work *= 2;
    // With few queries per row and a workgroup for most CUs the vector kernel reads at HBM's rate too.
    // Up to one per CU all of them end together, and at one or two queries the split kernel is the
    // slower one at any length (16 / 16 heads of 64, 12 x 4,096 tokens: 73 / 80; 32 / 16 of 64, 12 x
    // 2,149: 38 / 49; 16 x 4,096 of 16 / 16 heads 99 / 91); otherwise it needs a longer step for its
    // 9 us (12 / 4 of 64, 128 x 512 tokens: 29 / 31, x 1,024 55 / 53; 16 / 8 of 128, 64 x 512: 46 /
    // 50, x 1,024 105 / 93). Over 26,379 batches of 16-1,200 (sequence, kv head) pairs, lengths uniform
    // and ragged, the step taken is up to 7 times as fast as the vector kernel's and 3-8% slower in 10.
    const int64_t pairs = (int64_t)batch * num_heads / n_rep, cus = device_cus();
    if (nq == 1 ? 8 * pairs >= 3 * cus : 2 * pairs >= cus) {
        if (nq <= 2 && 2 * pairs >= cus && pairs < cus) return false;
        if (nq < 8 || pairs < cus) least *= 2;
    }
    return work >= least;
}

static int paged_decode_impl(void* out, int out_dtype, const void* q, const void* k_pool,
                             const void* v_pool, const int32_t* block_tables,
                             int max_blocks_per_seq, const int32_t* context_lens, int batch,
                             int num_heads, int kv_heads, int head_dim, int block_size,
                             int64_t num_slots, int max_context_len, float scale, int dtype,
                             void* workspace, size_t workspace_bytes, bool ws_from_scratch,
                             const int32_t* rows, const DecodeWs* fused, void* stream) {
    if (!valid_dtype(dtype) || !valid_dtype(out_dtype)) {
        set_error("paged_decode: unknown dtype (%d, out %d)", dtype, out_dtype);
        return FLOUR_ERR_INVALID_ARGUMENT;
    }
    if (batch < 0 || num_heads <= 0 || kv_heads <= 0 || num_heads % kv_heads != 0 ||
        head_dim <= 0 || block_size <= 0 || num_slots <= 0 || num_slots % block_size != 0 ||
        max_blocks_per_seq <= 0 || max_context_len < 0 ||
        (int64_t)max_context_len > (int64_t)max_blocks_per_seq * block_size) {
        set_error("paged_decode: bad shape (batch=%d heads=%d kv_heads=%d head_dim=%d bs=%d "
                  "num_slots=%lld max_blocks=%d max_ctx=%d)",
                  batch, num_heads, kv_heads, head_dim, block_size, (long long)num_slots,
                  max_blocks_per_seq, max_context_len);
        return FLOUR_ERR_INVALID_ARGUMENT;
    }
    if (batch == 0) return FLOUR_OK;
    if (!out || !q || !k_pool || !v_pool || !block_tables || !context_lens) {
        set_error("paged_decode: null pointer");
        return FLOUR_ERR_INVALID_ARGUMENT;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int n_rep = num_heads / kv_heads;
    const bool mfma = decode_mfma_supported(dtype, head_dim, block_size, n_rep, batch, num_heads,
                                            num_slots, q, k_pool, v_pool);
    if (!mfma && (rows || fused)) {
        set_error("paged_decode: row indices and the fused KV write need the matrix-core path");
        return FLOUR_ERR_UNSUPPORTED;
    }
    const int nwg = decode_workgroups(dtype);
    const size_t need = decode_ws_bytes(nwg, n_rep, head_dim, batch);
    const bool ws_ok = ws_from_scratch ? need <= DEC_SCRATCH_BYTES
                                       : workspace && workspace_bytes >= need &&
                                             ((uintptr_t)workspace % 256) == 0;
    // (an fp32 call without a workspace never touches the library's shared one)
    const bool f32_split =
        dtype == FLOUR_DTYPE_F32 &&
        decode_f32_split(head_dim, block_size, n_rep, batch, num_heads, num_slots, max_context_len,
                         out, q, k_pool, v_pool, ws_ok && !ws_from_scratch);
    if (!mfma && !f32_split) {
        // one query row per sequence: cu_seqlens == nullptr
        const int64_t qs = (int64_t)num_heads * head_dim;
        if (simt_supported(dtype, head_dim, q, qs, head_dim, k_pool, v_pool))
            return launch_attn_simt(dtype, out_dtype, out, qs, head_dim, q, qs, head_dim, k_pool,
                                    v_pool, nullptr, context_lens, block_tables,
                                    max_blocks_per_seq, batch, batch, num_heads, n_rep, head_dim,
                                    block_size, num_slots, max_context_len, scale, s);
        return launch_attn_generic(dtype, out_dtype, out, (int64_t)num_heads * head_dim, head_dim,
                                   q, (int64_t)num_heads * head_dim, head_dim, k_pool, v_pool,
                                   nullptr, context_lens, block_tables, max_blocks_per_seq, batch,
                                   batch, num_heads, n_rep, head_dim, block_size, num_slots,
                                   max_context_len, scale, s);
    }
    if (ws_from_scratch) {
        if (need > DEC_SCRATCH_BYTES) {
            set_error("paged_decode_noalloc: this call needs %zu bytes of split-context workspace, "
                      "more than the %zu bytes of the library's scratch; use "
                      "flour_hip_paged_decode with a caller workspace",
                      need, DEC_SCRATCH_BYTES);
            return FLOUR_ERR_WORKSPACE;
        }
        const int rc = scratch_for_current_device(&workspace);
        if (rc != FLOUR_OK) return rc;
        workspace_bytes = DEC_SCRATCH_BYTES;
    }
    if (!ws_ok) {
        set_error("paged_decode: workspace of %zu bytes (256-byte aligned) required, got %zu "
                  "at %p",
                  need, workspace_bytes, workspace);
        return FLOUR_ERR_WORKSPACE;
    }
    DecodeWs ws;
    ws.ml = static_cast<float*>(workspace);
    ws.o = reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                    align256((size_t)2 * nwg * n_rep * 2 * sizeof(float)));
    ws.pre = reinterpret_cast<int*>(
        reinterpret_cast<char*>(ws.o) +
        align256((size_t)2 * nwg * n_rep * (size_t)head_dim * sizeof(float)));
    ws.rows = rows;
    ws.xcd_w = g_xcd_weight;
    ws.k_new = fused ? fused->k_new : nullptr;
    ws.v_new = fused ? fused->v_new : nullptr;
    ws.new_st = fused ? fused->new_st : 0;
    ws.new_sh = fused ? fused->new_sh : 0;
    ws.new_slots = fused ? fused->new_slots : nullptr;
#define FLOUR_DEC(T)                                                                            \
    do {                                                                                        \
        if (out_dtype == FLOUR_DTYPE_F32)                                                       \
            return launch_decode_mfma<T, float>(head_dim, out, q, k_pool, v_pool, block_tables,           \
                                                max_blocks_per_seq, context_lens, batch,        \
                                                num_heads, kv_heads, n_rep, block_size,         \
                                                num_slots, max_context_len, scale, nwg, ws, s); \
        if (out_dtype == FLOUR_DTYPE_BF16)                                                      \
            return launch_decode_mfma<T, bf16_t>(head_dim, out, q, k_pool, v_pool, block_tables,          \
                                                 max_blocks_per_seq, context_lens, batch,       \
                                                 num_heads, kv_heads, n_rep, block_size,        \
                                                 num_slots, max_context_len, scale, nwg, ws,    \
                                                 s);                                            \
        return launch_decode_mfma<T, f16_t>(head_dim, out, q, k_pool, v_pool, block_tables,               \
                                            max_blocks_per_seq, context_lens, batch, num_heads, \
                                            kv_heads, n_rep, block_size, num_slots,             \
                                            max_context_len, scale, nwg, ws, s);                \
    } while (0)
    if (dtype == FLOUR_DTYPE_BF16) FLOUR_DEC(bf16_t);
    if (dtype == FLOUR_DTYPE_F32) FLOUR_DEC(float);
    FLOUR_DEC(f16_t);
#undef FLOUR_DEC
}

}  // namespace flour

namespace flour {

// Paged decode whose batch entry b reads q row rows[b] and writes out row rows[b] of a packed
// (rows, num_heads, head_dim) contiguous layout: the one-row sequences of a mixed
// continuous-batching step. Matrix-core shapes only (FLOUR_ERR_UNSUPPORTED otherwise, before
// any launch).
int paged_decode_rows(void* out, int out_dtype, const void* q, const void* k_pool,
                      const void* v_pool, const int32_t* block_tables, int max_blocks_per_seq,
                      const int32_t* context_lens, const int32_t* rows, int batch, int num_heads,
                      int kv_heads, int head_dim, int block_size, int64_t num_slots,
                      int max_context_len, float scale, int dtype, void* workspace,
                      size_t workspace_bytes, void* stream) {
    if (!rows) {
        set_error("paged_decode_rows: null row indices");
        return FLOUR_ERR_INVALID_ARGUMENT;
    }
    return paged_decode_impl(out, out_dtype, q, k_pool, v_pool, block_tables, max_blocks_per_seq,
                             context_lens, batch, num_heads, kv_heads, head_dim, block_size,
                             num_slots, max_context_len, scale, dtype, workspace, workspace_bytes,
                             false, rows, nullptr, stream);
}

int paged_decode_write_kv(void* out, int out_dtype, const void* q, void* k_pool, void* v_pool,
                          const int32_t* block_tables, int max_blocks_per_seq,
                          const int32_t* context_lens, int batch, int num_heads, int kv_heads,
                          int head_dim, int block_size, int64_t num_slots, int max_context_len,
                          float scale, int dtype, void* workspace, size_t workspace_bytes,
                          const void* k_new, const void* v_new, int64_t new_stride_tok,
                          int64_t new_stride_head, const int32_t* new_slots, void* stream) {
    const int es = (dtype == FLOUR_DTYPE_F32) ? 4 : 2;
    const uint64_t row_align = head_dim == 128 ? 16 : 8;  // a lane's share of a row
    // 16-token pages only: the fused instantiation for other page sizes spills registers in its
    // piece epilogue (a reload there waits for every chunk load in flight)
    if (!k_new || !v_new || !new_slots || batch < 1 || kv_heads <= 0 || block_size != 16 ||
        num_heads % kv_heads != 0 ||
        !decode_mfma_supported(dtype, head_dim, block_size, num_heads / kv_heads, batch,
                               num_heads, num_slots, q, k_pool, v_pool) ||
        (((uint64_t)(uintptr_t)k_new | (uint64_t)(uintptr_t)v_new |
          (uint64_t)(new_stride_tok * es) | (uint64_t)(new_stride_head * es)) &
         (row_align - 1)) != 0) {
        set_error("paged_decode_write_kv: shape not taken by the fused launch");
        return FLOUR_ERR_UNSUPPORTED;
    }
    DecodeWs fz{};
    fz.k_new = k_new;
    fz.v_new = v_new;
    fz.new_st = new_stride_tok;
    fz.new_sh = new_stride_head;
    fz.new_slots = new_slots;
    return paged_decode_impl(out, out_dtype, q, k_pool, v_pool, block_tables, max_blocks_per_seq,
                             context_lens, batch, num_heads, kv_heads, head_dim, block_size,
                             num_slots, max_context_len, scale, dtype, workspace, workspace_bytes,
                             false, nullptr, &fz, stream);
}

}  // namespace flour
