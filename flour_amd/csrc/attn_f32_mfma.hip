// attn_f32_mfma.hip — causal varlen prefill over fp32 pools on the fp32 matrix cores
// (v_mfma_f32_32x32x2_f32), head_dim 64 or 128. fp32 is the reference's model dtype when
// config.json names none (src/engine.rs:32-38); the arithmetic stays fp32 end to end: fp32
// products and sums in the matrix cores, fp32 softmax state.
//
// Semantics follow paged_attention (src/backend/cpu.rs:57-112): query row i of a sequence with
// q_len rows and kv_len cached positions sees kv position j iff j <= kv_len - q_len + i
// (cpu.rs:68, :88-95); query head h reads kv head h / n_rep (repeat_kv, cpu.rs:5-13); scores
// are q.k * scale; the softmax is folded online with a running max, sum and rescaled
// accumulator (cpu.rs:96-105); out = acc / sum (cpu.rs:111). A sequence with kv_len < q_len
// reads nothing and writes zero rows, as the other paths of this library do.
//
// Work: one workgroup per (query head, sequence, tile of 32 query rows), tiles of the highest
// index first (they read the longest kv ranges). Its W waves split the tile's causal kv range
// in steps of 32 positions (wave w takes steps w, w + W, ...) and fold their partial states
// together at the end through LDS, by log-sum-exp.
//
// Per step, with lane l holding query row r = l % 32 and half h = l / 32:
//  * S^T = K Q^T (32 positions x 32 rows) over D/2 products of k = 2: product s pairs head-dim
//    element D/2 h + s of the position (A, lane l: position l % 32) and of the row (B, lane l:
//    row l % 32), so each lane reads one contiguous half-row of K and of Q.
//  * The result leaves lane l with the scores of row r at positions 8 (e / 4) + 4 h + e % 4,
//    e = 0 .. 15: the row's max and sum need only the partner lane l ^ 32.
//  * O^T += V^T P^T over 16 products of k = 2, one per score register: product s takes the
//    lane's own score s as its B operand (position 8 (s / 4) + 4 h + s % 4, row r), and V at
//    that position as A, at head-dim element D/32 c + t of output tile t for lane row c = l % 32.
//    Each lane so reads D/32 contiguous elements of one V row per product; the positions' pool
//    slots come from the lanes that hold them for K (lane shuffles, no second table walk).
#include <math.h>

#include "flour_common.h"
#include "prefill_items.h"

namespace flour {

static constexpr int F32M_QT = 32;  // query rows per workgroup
static constexpr int F32M_KT = 32;  // kv positions per step
// Waves per workgroup: at head_dim 64 a wave holds 128 registers (two per SIMD, and two
// workgroups per CU); at 128 it holds 256, one per SIMD (8 waves of ~200 registers measured
// slower).
__host__ __device__ constexpr int f32m_waves(int d) { return d == 64 ? 8 : 4; }

__device__ __forceinline__ f32x16 mfma32x32x2_f32(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

template <int D>
__global__ __launch_bounds__(f32m_waves(D) * 64) void prefill_f32_mfma_kernel(
    void* __restrict__ out, int out_dtype, int64_t o_st, int64_t o_sh,
    const float* __restrict__ q, int64_t q_st, int64_t q_sh, const float* __restrict__ k_pool,
    const float* __restrict__ v_pool, const int32_t* __restrict__ cu_seqlens_q,
    const int32_t* __restrict__ q_rows, const int32_t* __restrict__ kv_lens,
    const int32_t* __restrict__ block_tables, int max_blocks, int n_rep, int block_size,
    int num_slots, int n_qt, float scale_log2) {
    constexpr int W = f32m_waves(D);
    constexpr int DH = D / 2;   // products of S^T per step
    constexpr int DT = D / 32;  // 32-row tiles of O^T
    constexpr int NS = 16 * DT + 2;  // a lane's state: O^T registers, max, sum
    // partial states of the upper half of the waves still merging, [wave][value][lane]
    __shared__ float red[(W / 2) * NS * 64];

    const int head = blockIdx.x, s = blockIdx.y, qt = n_qt - 1 - (int)blockIdx.z;
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const int r = lane & 31, h = lane >> 5;
    const int c0 = cu_seqlens_q[s];
    const int q_len = cu_seqlens_q[s + 1] - c0;
    if (qt * F32M_QT >= q_len) return;  // uniform: no such tile in this sequence
    const int row0 = q_rows ? q_rows[s] : c0;  // the sequence's first packed row
    const int kv_len = min(kv_lens[s], max_blocks * block_size);
    const int off = kv_len - q_len;  // row i sees positions j <= off + i
    const int i = qt * F32M_QT + r;  // this lane's row in the sequence
    const int last = min(qt * F32M_QT + F32M_QT, q_len) - 1;
    const int kv_end = kv_len >= q_len ? off + last + 1 : 0;  // positions the tile reads
    const int lim = (i < q_len && kv_len >= q_len) ? off + i : -1;
    const int kvh = head / n_rep;
    const int32_t* bt = block_tables + (int64_t)s * max_blocks;
    const int max_phys = num_slots / block_size - 1;
    const float* kbase = k_pool + (int64_t)kvh * num_slots * D;
    const float* vbase = v_pool + (int64_t)kvh * num_slots * D;

    // this lane's half-row of Q (rows past the sequence read its last row; they are masked),
    // pre-scaled into the exp2 domain
    float qv[DH];
    {
        const float* qp = q + (int64_t)(row0 + min(i, q_len - 1)) * q_st + (int64_t)head * q_sh + DH * h;
#pragma unroll
        for (int x = 0; x < DH / 4; x++) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(qp + 4 * x);
#pragma unroll
            for (int e = 0; e < 4; e++) qv[4 * x + e] = v[e] * scale_log2;
        }
    }

    float m = -INFINITY, l = 0.0f;
    f32x16 o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) o[t][e] = 0.0f;

    const int n_st = (kv_end + F32M_KT - 1) / F32M_KT;
    for (int st = w; st < n_st; st += W) {
        const int kv0 = st * F32M_KT;
        // pool slot of position kv0 + r (row 0 past the tile's range: those scores are masked);
        // a block id outside the pool is clamped into it
        int slot = 0;
        {
            const int j = kv0 + r;
            if (j < kv_end) {
                const int lb = j / block_size;
                const int id = bt[lb];
                const int phys = id < 0 ? 0 : (id > max_phys ? max_phys : id);
                slot = phys * block_size + (j - lb * block_size);
            }
        }
        float kx[DH];
        {
            const float* kp = kbase + (int64_t)slot * D + DH * h;
#pragma unroll
            for (int x = 0; x < DH / 4; x++) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(kp + 4 * x);
#pragma unroll
                for (int e = 0; e < 4; e++) kx[4 * x + e] = v[e];
            }
        }
        // V at the positions of this lane's scores; the slot of position 8 (e/4) + 4h + e%4 is
        // held by that lane
        float vx[16][DT];
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int src = 8 * (e >> 2) + 4 * h + (e & 3);
            const int sl = __shfl(slot, src, 64);
            const float* vp = vbase + (int64_t)sl * D + DT * r;
            if constexpr (DT == 4) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(vp);
#pragma unroll
                for (int t = 0; t < 4; t++) vx[e][t] = v[t];
            } else {
                const f32x2 v = *reinterpret_cast<const f32x2*>(vp);
                vx[e][0] = v[0];
                vx[e][1] = v[1];
            }
        }
        // S^T = K Q^T
        f32x16 sc;
#pragma unroll
        for (int e = 0; e < 16; e++) sc[e] = 0.0f;
#pragma unroll
        for (int x = 0; x < DH; x++) sc = mfma32x32x2_f32(kx[x], qv[x], sc);
        // causal mask and the row's max (lanes l and l ^ 32 hold the same row)
        float tm = -INFINITY;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            const int j = kv0 + 8 * (e >> 2) + 4 * h + (e & 3);
            if (j > lim) sc[e] = -INFINITY;
            tm = fmaxf(tm, sc[e]);
        }
        tm = max_across_halves(tm);
        const float m_new = fmaxf(m, tm);
        const float mu = m_new == -INFINITY ? 0.0f : m_new;  // nothing visible yet: all p = 0
        const float alpha = fast_exp2(m - mu);
        m = m_new;
        float p[16], ps = 0.0f;
#pragma unroll
        for (int e = 0; e < 16; e++) {
            p[e] = fast_exp2(sc[e] - mu);
            ps += p[e];
        }
        l = l * alpha + ps;
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) o[t][e] *= alpha;
        // O^T += V^T P^T
#pragma unroll
        for (int e = 0; e < 16; e++)
#pragma unroll
            for (int t = 0; t < DT; t++) o[t] = mfma32x32x2_f32(vx[e][t], p[e], o[t]);
    }
    l = sum_across_halves(l);  // the row's sum over both halves of its positions

    // fold the waves' states pairwise: the upper half writes, the lower half merges
#pragma unroll
    for (int half = W / 2; half >= 1; half >>= 1) {
        if (w >= half && w < 2 * half) {
            float* dst = red + (w - half) * NS * 64 + lane;
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int e = 0; e < 16; e++) dst[(16 * t + e) * 64] = o[t][e];
            dst[16 * DT * 64] = m;
            dst[(16 * DT + 1) * 64] = l;
        }
        __syncthreads();
        if (w < half) {
            const float* src = red + w * NS * 64 + lane;
            const float mb = src[16 * DT * 64], lb = src[(16 * DT + 1) * 64];
            const float mm = fmaxf(m, mb);
            const float mz = mm == -INFINITY ? 0.0f : mm;
            const float fa = fast_exp2(m - mz), fb = fast_exp2(mb - mz);
            l = l * fa + lb * fb;
            m = mm;
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int e = 0; e < 16; e++) o[t][e] = o[t][e] * fa + src[(16 * t + e) * 64] * fb;
        }
        if (half > 1) __syncthreads();
    }
    if (w != 0 || i >= q_len) return;
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;  // no visible position: a zero row
    const int64_t obase = (int64_t)(row0 + i) * o_st + (int64_t)head * o_sh;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        float v[DT];
#pragma unroll
        for (int t = 0; t < DT; t++) v[t] = o[t][e] * inv;
        store_run<DT>(out, out_dtype, obase + DT * (8 * (e >> 2) + 4 * h + (e & 3)), v);
    }
}

// ---- Larger batches. An item is (kv head, group of HW query heads, sequence, 32 (4 / HW) query
// rows), HW = 4, 2 or 1, for a workgroup of eight waves: waves w and w + 4, which share a SIMD, own
// the same 32 rows of one head and take alternate 32-position tiles; their states are folded at
// the end. K / V rows go straight into LDS, once for all eight waves (double-buffered, one barrier
// per step of 64 positions, 128 at D 64, loads one step ahead and block ids two), where the kernel
// above has every wave gather its own from L2 with nothing in flight under its products. Bound by
// the fp32 matrix cores: a wave's tile is D products of 64 cycles.
//  * One workgroup per CU takes items longest first, as a snake over the list: left to the
//    dispatcher, workgroups of this size fill the CUs in a fixed rotation and a ragged batch waits
//    for the unluckiest (8 x U[300, 1,024] rows, 32 / 8 heads of 128: 461 us, dealt 352).
//  * The first four waves run at raised priority and a wave keeps two chains of products going, so
//    that a SIMD's second wave has its products left for the time of the first's softmax.
//  * S^T as above, the 16-byte chunk c of K row r at chunk c ^ (r % 16) (conflict-free reads).
//  * O^T tile t holds dims 32 t .. 32 t + 31: its A operand is V[position][32 t + lane % 32], a
//    4-byte read of a V row, so V needs no transpose.
//  * fp32 sums are kept short (chains of 32 products for a score, of the tile's 32 positions for
//    an output, then sums of those): error against 64 bits 1.4-2.4e-7 over 25 batches, where the
//    kernel above has 2.2-5.1e-7.
// Against the kernel above: 8 x U[256, 1,024] rows, 32 / 8 heads of 128, 429 -> 346 us (82
// TFLOP/s); 16 x 512 552 -> 414; 1 x 4,096 1,327 -> 1,181 (116); 32 x U[256, 400], 14 / 2 heads of
// 64, 153 -> 112.
static constexpr int F32T_SPLIT = 2;  // waves per (head, row block)
static constexpr int F32T_WAVES = 4 * F32T_SPLIT;
static constexpr uint32_t F32T_OOR = 0x80000000u;  // buffer offset past any pool: loads read 0
template <int D, bool BS16>
__global__ __launch_bounds__(F32T_WAVES * 64, 2) void prefill_f32_tile_kernel(
    void* __restrict__ out, int out_dtype, int64_t o_st, int64_t o_sh,
    const float* __restrict__ q, int64_t q_st, int64_t q_sh, const float* __restrict__ k_pool,
    const float* __restrict__ v_pool, const int32_t* __restrict__ cu_seqlens_q,
    const int32_t* __restrict__ kv_lens, const int32_t* __restrict__ block_tables, int max_blocks,
    int num_seqs, int kv_heads, int n_rep, int hw, int block_size, int num_slots, int n_qt,
    float scale_log2) {
    constexpr int DH = D / 2, DT = D / 32;
    constexpr int SUB = 128 / D;              // 32-position tiles per wave and step
    constexpr int KT = F32M_KT * F32T_SPLIT * SUB;  // positions per step
    constexpr int CPR = D / 4;                // 16-byte chunks per row
    constexpr int RPL = 64 / CPR;             // rows per wave load of 1 KB
    constexpr int NP = KT / (RPL * F32T_WAVES);  // loads per wave, step and pool (4 at D 128)
    constexpr int NS = 16 * DT + 2;           // a lane's state: O^T registers, max, sum
    __shared__ __attribute__((aligned(16))) float lds[4 * KT * D];
    static_assert(4 * (F32T_SPLIT - 1) * NS * 64 <= 4 * KT * D, "the states fit the tiles");
    __shared__ ItemSeq seqs[64];
    auto kt = [&](int buf) { return lds + buf * KT * D; };
    auto vt = [&](int buf) { return lds + (2 + buf) * KT * D; };

    const int groups = (n_rep + hw - 1) / hw, per_row = kv_heads * groups;
    const int rows = F32M_QT * (4 / hw);  // query rows of an item
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = lane & 31, h = lane >> 5;
    const int wq = w & 3, ks = w >> 2;  // (head, row block), part of each step
    const int max_phys = num_slots / block_size - 1;
    const uint32_t head_bytes = (uint32_t)num_slots * D * 4u;
    const int G = gridDim.x;

    using Walk = ItemWalk<true>;
    Walk items;
    items.start(cu_seqlens_q, kv_lens, num_seqs, max_blocks * block_size, rows, n_qt, per_row, lane,
                seqs);
    if (ks == 0) __builtin_amdgcn_s_setprio(1);

    for (int round = 0;; round++) {
        int s, qt, x;
        ItemSeq sq;
        if (!items.find(Walk::deal(round, G, blockIdx.x), lane, s, sq, qt, x)) break;
        const int kvh = x / groups, h0 = (x - kvh * groups) * hw;
        const int c0 = sq.c0;
        const int q_len = sq.rows;
        const int kv_len = sq.kv;
        const int off = kv_len - q_len;  // row i sees positions j <= off + i
        const bool reads = kv_len >= q_len;
        const int kv_end = reads ? off + min(qt * rows + rows, q_len) : 0;  // the item's range
        const int hl = h0 + wq % hw;
        const int i0 = qt * rows + F32M_QT * (wq / hw);  // the wave's first row
        const bool active = hl < n_rep && i0 < q_len;    // uniform over the wave
        const int i = i0 + r;
        const int head = kvh * n_rep + min(hl, n_rep - 1);
        const int lim = (active && i < q_len && reads) ? off + i : -1;
        const int w_end = active && reads ? off + min(i0 + F32M_QT, q_len) : 0;  // the wave's range
        const int w_full = off + i0;  // positions up to here are visible to every row of the wave
        const int32_t* bt = block_tables + (int64_t)s * max_blocks;
        const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(k_pool + (int64_t)kvh * num_slots * D), (short)0, (int)head_bytes, BUF_DWORD3);
        const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(v_pool + (int64_t)kvh * num_slots * D), (short)0, (int)head_bytes, BUF_DWORD3);

        float qv[DH];
        {
            const float* qp =
                q + (int64_t)(c0 + min(i, q_len - 1)) * q_st + (int64_t)head * q_sh + DH * h;
#pragma unroll
            for (int y = 0; y < DH / 4; y++) {
                const f32x4 v = *reinterpret_cast<const f32x4*>(qp + 4 * y);
#pragma unroll
                for (int e = 0; e < 4; e++) qv[4 * y + e] = v[e] * scale_log2;
            }
        }

        // Staging, straight into LDS: load p of wave w fills rows srow + RPL F32T_WAVES p of the
        // step, lane l chunk l % CPR of row l / CPR. A K row's chunk c sits at chunk c ^ (row % 16)
        // (conflict-free fragment reads), so the lane reads that chunk of the row; V as it is.
        const int lrow = lane / CPR, lchunk = lane % CPR;
        const int srow = RPL * w + lrow;
        auto load_ids = [&](int kv0, int* ids) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < NP; p++) {
                const int j = min(kv0 + srow + RPL * F32T_WAVES * p, max(kv_end - 1, 0));
                ids[p] = bt[BS16 ? j >> 4 : j / block_size];
            }
        };
        auto load_tile = [&](int kv0, const int* ids, int buf) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < NP; p++) {
                const int row = srow + RPL * F32T_WAVES * p, j = kv0 + row;
                const int in = BS16 ? j & 15 : j % block_size;
                const int phys = min(max(ids[p], 0), max_phys);  // a bad block id stays in the pool
                const uint32_t at = (uint32_t)(phys * block_size + in) * (uint32_t)(4 * D);
                const bool there = j < kv_end;  // rows past the range read zeros (masked anyway)
                const uint32_t dst = (uint32_t)(RPL * (w + F32T_WAVES * p)) * (uint32_t)(4 * D);
                dma_b128(there ? at + 16u * (uint32_t)(lchunk ^ (row & 15)) : F32T_OOR, k_rsrc,
                         lds_byte_addr(kt(buf)) + dst, 0u);
                dma_b128(there ? at + 16u * (uint32_t)lchunk : F32T_OOR, v_rsrc,
                         lds_byte_addr(vt(buf)) + dst, 0u);
            }
        };

        float m = -INFINITY, l = 0.0f;
        f32x16 o[DT];
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) o[t][e] = 0.0f;

        const int n_st = (kv_end + KT - 1) / KT;
        int ids[NP];
        load_ids(0, ids);
        __syncthreads();  // the last item's states are read
        if (n_st > 0) {
            load_tile(0, ids, 0);
            load_ids(KT, ids);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        for (int st = 0; st < n_st; st++) {
            const int buf = st & 1;
            if (st + 1 < n_st) {
                load_tile((st + 1) * KT, ids, buf ^ 1);
                load_ids((st + 2) * KT, ids);
            }
#pragma unroll
            for (int u = 0; u < SUB; u++) {
                const int row0 = F32M_KT * (ks + F32T_SPLIT * u);  // the wave's tile in the step
                const int kv0 = st * KT + row0;
                if (kv0 >= w_end) continue;  // uniform over the wave
                const float* kr = kt(buf) + (row0 + r) * D;
                f32x16 sc;
                // two chains of 32 products (16 steps of k = 2) at a time: independent products
                // keep the matrix core busy from one wave
#pragma unroll
                for (int c = 0; c < DH / 32; c++) {
                    f32x16 pa, pb;
#pragma unroll
                    for (int e = 0; e < 16; e++) pa[e] = pb[e] = 0.0f;
#pragma unroll
                    for (int y = 0; y < 4; y++) {
                        // chunk DH / 4 h + 8c + y (+ 4) of the row
                        const int ca = (DH / 4) * h + 8 * c + y;
                        const f32x4 ka = *reinterpret_cast<const f32x4*>(kr + 4 * (ca ^ (r & 15)));
                        const f32x4 kb = *reinterpret_cast<const f32x4*>(kr + 4 * ((ca + 4) ^ (r & 15)));
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            pa = mfma32x32x2_f32(ka[e], qv[32 * c + 4 * y + e], pa);
                            pb = mfma32x32x2_f32(kb[e], qv[32 * c + 16 + 4 * y + e], pb);
                        }
                    }
                    if (c == 0)
                        sc = pa + pb;
                    else
                        sc += pa + pb;
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (kv0 + F32M_KT - 1 > w_full) {  // the tile crosses some row's limit
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        if (kv0 + 8 * (e >> 2) + 4 * h + (e & 3) > lim) sc[e] = -INFINITY;
                }
                float tm = sc[0];
#pragma unroll
                for (int e = 1; e < 16; e++) tm = fmaxf(tm, sc[e]);
                tm = max_across_halves(tm);
                const float m_new = fmaxf(m, tm);
                const float mu = m_new == -INFINITY ? 0.0f : m_new;  // nothing visible: all p = 0
                const float alpha = fast_exp2(m - mu);
                m = m_new;
                float ps = 0.0f;
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    sc[e] = fast_exp2(sc[e] - mu);
                    ps += sc[e];
                }
                l = l * alpha + ps;
                const float* vr = vt(buf) + (row0 + 4 * h) * D + r;
#pragma unroll
                for (int t = 0; t < DT; t += 2) {
                    f32x16 pa, pb;
#pragma unroll
                    for (int e = 0; e < 16; e++) pa[e] = pb[e] = 0.0f;
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        const float* v = vr + (8 * (e >> 2) + (e & 3)) * D + 32 * t;
                        pa = mfma32x32x2_f32(v[0], sc[e], pa);
                        pb = mfma32x32x2_f32(v[32], sc[e], pb);
                    }
#pragma unroll
                    for (int e = 0; e < 16; e++) o[t][e] = fmaf(o[t][e], alpha, pa[e]);
#pragma unroll
                    for (int e = 0; e < 16; e++) o[t + 1][e] = fmaf(o[t + 1][e], alpha, pb[e]);
                }
            }
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the next step's rows are in LDS
            __syncthreads();
        }
        l = sum_across_halves(l);
        // fold the two waves' states (the last step's barrier is behind every read of the tiles)
        if (ks) {
            float* dst = lds + wq * NS * 64 + lane;
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int e = 0; e < 16; e++) dst[(16 * t + e) * 64] = o[t][e];
            dst[16 * DT * 64] = m;
            dst[(16 * DT + 1) * 64] = l;
        }
        __syncthreads();
        if (!ks && active && i < q_len) {
            const float* src = lds + wq * NS * 64 + lane;
            const float mb = src[16 * DT * 64], lb = src[(16 * DT + 1) * 64];
            const float mm = fmaxf(m, mb);
            const float mz = mm == -INFINITY ? 0.0f : mm;
            const float fa = fast_exp2(m - mz), fb = fast_exp2(mb - mz);
            l = l * fa + lb * fb;
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;  // no visible position: a zero row
            const int64_t obase = (int64_t)(c0 + i) * o_st + (int64_t)head * o_sh + 4 * h;
#pragma unroll
            for (int t = 0; t < DT; t++)
#pragma unroll
                for (int e = 0; e < 16; e += 4) {
                    float v[4];
#pragma unroll
                    for (int y = 0; y < 4; y++)
                        v[y] = (o[t][e + y] * fa + src[(16 * t + e + y) * 64] * fb) * inv;
                    store_run<4>(out, out_dtype, obase + 32 * t + 2 * e, v);
                }
        }
    }
}

// 0: the vector kernel, 1: by the rules below, 2 / 3: never / always (within its limits) the tile
// kernel. A test / tuning switch.
static int g_prefill_f32_mfma = 1;

bool prefill_f32_mfma_supported(int dtype, int head_dim, int num_seqs, int max_seqlen_q,
                                int block_size, int64_t num_slots) {
    const int64_t n_qt = ((int64_t)max_seqlen_q + F32M_QT - 1) / F32M_QT;
    return g_prefill_f32_mfma && dtype == FLOUR_DTYPE_F32 && (head_dim == 64 || head_dim == 128) &&
           num_seqs <= 65535 && n_qt <= 65535 && block_size > 0 && num_slots <= 0x7fffffff &&
           num_slots % block_size == 0;
}

// The caller checks prefill_f32_mfma_supported, the 16-byte alignment of q, the pools and out
// and of their row and head strides. kv_cap bounds the kv lengths (for the choice of the kernel).
int launch_prefill_f32_mfma(int out_dtype, void* out, int64_t o_st, int64_t o_sh, const void* q,
                            int64_t q_st, int64_t q_sh, const void* k_pool, const void* v_pool,
                            const int32_t* cu_seqlens_q, const int32_t* q_rows,
                            const int32_t* kv_lens, const int32_t* block_tables, int max_blocks,
                            int num_seqs, int max_seqlen_q, int total_q, int64_t kv_cap,
                            int num_heads, int n_rep, int head_dim, int block_size,
                            int64_t num_slots, float scale, hipStream_t stream) {
    const int n_qt = (max_seqlen_q + F32M_QT - 1) / F32M_QT;
    if (n_qt == 0 || num_seqs == 0) return FLOUR_OK;
    const dim3 grid((unsigned)num_heads, (unsigned)num_seqs, (unsigned)n_qt);
    const float sl2 = scale * 1.4426950408889634f;
    // Which batches run on the tile kernel. Its items are larger and split over two waves instead of
    // four or eight, so it needs enough of them, none that outlasts the rest, and full ones. Measured,
    // other / tile in us:
    //  * Items per CU, counted from the batch's rows: 32 / 8 heads of 128, 1 x 1,024 rows (1) 120 /
    //    157, 2 x 1,024 (2) 203 / 168; 14 / 2 of 64, whose groups of four leave a slot without a head,
    //    1 x 6,190 (3.0) 697 / 758. From 2.5, 4 with such a slot or with 128-row items.
    //  * Rows per sequence: 16 / 16 of 128 (128-row items), 32 x 132 rows 94 / 143, 32 x 324 325 / 354,
    //    8 x 1,296 848 / 742. At least 64, 128 and 640.
    //  * The longest item that kv_cap (the block table's width, if no better) allows, since the host
    //    cannot tell one long context from a cached prefix of all: up to 1.5 times a CU's share of the
    //    rows' own causal ranges. 28 / 4 of 128, 64 x 42 rows, one behind 4,096 tokens 308 / 610; 32 /
    //    8 of 128, 1 x 2,075 behind 2,048 1,096 / 1,175.
    // Of 21,095 batches with and without prefixes, some of one sequence alone, this takes 7,337: 7 of
    // them are more than 3% slower than on the other kernel, the geometric mean is 1.24x.
    // Its item list holds up to 64 sequences, its loads 32-bit offsets.
    const int hw = item_heads(n_rep), kv_heads = num_heads / n_rep;
    const int rows = F32M_QT * (4 / hw);
    const int64_t per_row = (int64_t)kv_heads * ((n_rep + hw - 1) / hw);
    const int64_t cus = device_cus();
    const bool fits = !q_rows && num_seqs <= 64 && num_slots * head_dim * 4 <= 0x7fffffff &&
                      per_row * num_seqs * ((int64_t)max_seqlen_q / rows + 1) <= 0x3fffffff;
    const int64_t full = per_row * (total_q / rows);  // items of full tiles
    const bool spare = n_rep % hw != 0;               // slots without a head
    const int mean = total_q / num_seqs;
    const bool wanted = 2 * full >= (spare || rows == 128 ? 8 : 5) * cus &&
                        mean >= (rows == 128 ? 640 : spare ? 128 : 64) &&
                        4 * kv_cap * cus <= 3 * full * mean;
    const bool tiled =
        fits && g_prefill_f32_mfma != 2 && (g_prefill_f32_mfma == 3 || wanted);
    if (tiled) {
        const int nt = (max_seqlen_q + rows - 1) / rows;
        auto kern = head_dim == 64 ? (block_size == 16 ? prefill_f32_tile_kernel<64, true>
                                                       : prefill_f32_tile_kernel<64, false>)
                                   : (block_size == 16 ? prefill_f32_tile_kernel<128, true>
                                                       : prefill_f32_tile_kernel<128, false>);
        kern<<<dim3((unsigned)cus), dim3(F32T_WAVES * 64), 0, stream>>>(
            out, out_dtype, o_st, o_sh, static_cast<const float*>(q), q_st, q_sh,
            static_cast<const float*>(k_pool), static_cast<const float*>(v_pool), cu_seqlens_q,
            kv_lens, block_tables, max_blocks, num_seqs, kv_heads, n_rep, hw, block_size,
            (int)num_slots, nt, sl2);
        return check_hip(hipGetLastError(), "varlen_prefill (fp32 matrix cores) launch");
    }
#define FLOUR_F32M(D)                                                                            \
    prefill_f32_mfma_kernel<D><<<grid, dim3(f32m_waves(D) * 64), 0, stream>>>(                   \
        out, out_dtype, o_st, o_sh, static_cast<const float*>(q), q_st, q_sh,                    \
        static_cast<const float*>(k_pool), static_cast<const float*>(v_pool), cu_seqlens_q,      \
        q_rows, kv_lens, block_tables, max_blocks, n_rep, block_size, (int)num_slots, n_qt, sl2)
    if (head_dim == 64)
        FLOUR_F32M(64);
    else
        FLOUR_F32M(128);
#undef FLOUR_F32M
    return check_hip(hipGetLastError(), "varlen_prefill (fp32 matrix cores) launch");
}

}  // namespace flour

using namespace flour;

// fp32 prefill at head_dim 64 / 128: 1 (the default) on the fp32 matrix cores, 0 on the vector
// kernel; 2 and 3 as 1, but never / always, within its limits, on the tile kernel. A test / tuning
// switch.
extern "C" int flour_hip_set_prefill_f32_mfma(int mode) {
    if (mode < 0 || mode > 3) {
        set_error("set_prefill_f32_mfma: mode %d is not 0 to 3", mode);
        return FLOUR_ERR_INVALID_ARGUMENT;
    }
    g_prefill_f32_mfma = mode;
    return FLOUR_OK;
}
