// prefill_thin.hip — causal varlen prefill of small batches over 16-bit pools at head_dim 64 on
// gfx950 matrix cores: one prompt, a few short ones, the prompts of a mixed step.
//
// Semantics follow paged_attention (src/backend/cpu.rs:57-112) as in varlen_prefill.hip: query row
// i of a sequence with q_len rows and kv_len cached positions sees kv position j iff j <= kv_len -
// q_len + i (cpu.rs:68, :88-95); query head h reads kv head h / n_rep (repeat_kv, cpu.rs:5-13); a
// sequence with kv_len < q_len reads nothing and writes zero rows.
//
// varlen_prefill.hip's items are 128 query rows x 2 heads: a small batch has fewer of them than the
// chip has CUs and waits for one item's chain of kv tiles. Here an item is SLOTS = 4 or 2 (head,
// 32-row block) slots of one kv head and sequence, each on 8 / SLOTS waves that take every 2nd or
// 4th 32-position tile: two to eight times the items, and a chain half or a quarter as long. The
// price is that K / V are staged for fewer rows at a time.
//  * One workgroup per CU walks the items longest first (prefill_items.h). The K / V rows of step
//    t + 1 are requested before step t is computed, then written to the other LDS buffer (K rows of D
//    + 8 elements; V transposed, token t at column sigma16(t), rows of a step's positions + 8): one
//    barrier a step; block ids two steps ahead.
//  * As built, a step still waits for those rows: the wait for Q's own loads, which the compiler puts
//    at their first use inside the step loop, counts the step's loads too (vmcnt(3) .. (0) before the
//    four score products). A step is therefore bound by one memory round trip and the vector issue
//    behind it (exp2, packing, the split of P), and the batch by its longest chain of steps.
//  * S^T = K Q^T and O^T = V^T P^T on v_mfma_f32_32x32x16, the score registers being the B operand
//    of the second product after 16-bit packing (varlen_prefill.hip has the layouts). Over bf16 pools
//    P is split into hi + lo bf16 parts, two products each, with V as stored: ~16 bits of P and no
//    range limits, so no item is computed twice. Over f16 pools P is rounded once to f16, as there.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "flour_common.h"
#include "prefill_items.h"

namespace flour {

static constexpr int PT_D = 64;    // head_dim
static constexpr int PT_WAVES = 8;  // SLOTS (head, row block) x SPLIT shares of each step
static constexpr uint32_t PT_OOR = 0x80000000u;  // buffer offset past any pool: loads read 0

template <typename T, bool BS16, int SLOTS>
__global__ __launch_bounds__(PT_WAVES * 64, 2) void prefill_thin_kernel(
    void* __restrict__ out, int out_dtype, int64_t o_st, int64_t o_sh, const T* __restrict__ q,
    int64_t q_st, int64_t q_sh, const T* __restrict__ k_pool, const T* __restrict__ v_pool,
    const int32_t* __restrict__ cu_seqlens, const int32_t* __restrict__ q_rows,
    const int32_t* __restrict__ kv_lens, const int32_t* __restrict__ block_tables, int max_blocks,
    int num_seqs, int kv_heads, int n_rep, int hw, int block_size, int64_t num_slots, int n_qt,
    float scale_log2) {
    constexpr int D = PT_D, SPLIT = PT_WAVES / SLOTS;
    constexpr int SUB = SPLIT == 2 ? 2 : 1;  // 32-position tiles per wave and step
    constexpr int KT = 32 * SPLIT * SUB;  // positions per step
    constexpr int VP = KT + 8;         // elements per V^T row in LDS
    constexpr int KP = D + 8;          // elements per K row in LDS
    constexpr int NKQ = D / 16;        // 16-dim k-steps of S^T
    constexpr int NMT = D / 32;        // 32-dim blocks of O^T
    constexpr int CPR = D / 8;         // 16-byte chunks per row
    constexpr int RPP = PT_WAVES * 64 / CPR;  // K rows per staging pass
    constexpr int KPASS = KT / RPP;
    constexpr int VPASS = (KT / 2) * CPR / (PT_WAVES * 64);  // V token pairs per thread
    constexpr int NS = 16 * NMT + 2;   // a lane's state: O^T registers, max, sum
    constexpr bool HILO = std::is_same<T, bf16_t>::value;
    constexpr int BUF = KT * KP + D * VP;  // elements
    constexpr int LDS_BYTES = std::max(2 * BUF * 2, (SPLIT - 1) * SLOTS * NS * 64 * 4);
    __shared__ __attribute__((aligned(16))) uint8_t lds[LDS_BYTES];
    auto kt = [&](int buf) { return reinterpret_cast<uint16_t*>(lds) + buf * BUF; };
    auto vt = [&](int buf) { return reinterpret_cast<uint16_t*>(lds) + buf * BUF + KT * KP; };

    const int groups = (n_rep + hw - 1) / hw;
    const int rows = 32 * (SLOTS / hw);  // query rows of an item
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = lane & 31, h2 = lane >> 5;
    const int wq = w % SLOTS, ks = w / SLOTS;  // (head, row block), share of each step
    const int max_phys = (int)(num_slots / block_size - 1);
    const uint32_t head_bytes = (uint32_t)(num_slots * D * (int64_t)sizeof(T));
    constexpr uint32_t ROW_BYTES = D * sizeof(T);
    // staging: K chunk tid % CPR of rows tid / CPR + RPP p; V tokens 2 vp, 2 vp + 1 (vp = tid % RPP +
    // RPP p), dims v_col .. + 7: lanes of a wave hold consecutive token pairs, so that its V^T writes
    // are runs of a row (conflict-free)
    const int k_row = tid / CPR, k_col = (tid % CPR) * 8;
    const int v_tp = tid % RPP, v_col = (tid / RPP) * 8;

    using Walk = ItemWalk<false>;
    Walk items;
    items.start(cu_seqlens, kv_lens, num_seqs, max_blocks * block_size, rows, n_qt,
                kv_heads * groups, lane);
    for (int round = 0;; round++) {
        int s, qt, x;
        ItemSeq sq;
        if (!items.find(Walk::deal(round, gridDim.x, blockIdx.x), lane, s, sq, qt, x)) break;
        const int kvh = x / groups, h0 = (x - kvh * groups) * hw;
        const int c0 = sq.c0;
        const int q_len = sq.rows;
        const int kv_len = sq.kv;
        const int row0 = q_rows ? __builtin_amdgcn_readfirstlane(q_rows[s]) : c0;
        const int off = kv_len - q_len;  // row i sees positions j <= off + i
        const bool reads = kv_len >= q_len;
        const int kv_end = reads ? off + min(qt * rows + rows, q_len) : 0;  // the item's range
        const int hl = h0 + wq % hw;
        const int i0 = qt * rows + 32 * (wq / hw);     // the wave's first row
        const bool active = hl < n_rep && i0 < q_len;  // uniform over the wave
        const int i = i0 + r;
        const int head = kvh * n_rep + min(hl, n_rep - 1);
        const int lim = off + min(i, q_len - 1);  // rows past the sequence repeat its last
        const int w_end = active && reads ? off + min(i0 + 32, q_len) : 0;  // the wave's range
        const int w_full = off + i0;  // positions up to here are visible to every row of the wave
        const int32_t* bt = block_tables + (int64_t)s * max_blocks;
        const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(k_pool + (int64_t)kvh * num_slots * D), (short)0, (int)head_bytes, BUF_DWORD3);
        const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(v_pool + (int64_t)kvh * num_slots * D), (short)0, (int)head_bytes, BUF_DWORD3);

        // block ids of the thread's K rows and V token pairs (a pair lies in one page)
        const int kv_last = max(kv_end - 1, 0);
        constexpr int NID = KPASS + VPASS;
        auto load_ids = [&](int kv0, int* ids) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < NID; p++) {
                const int j = min(kv0 + (p < KPASS ? k_row + RPP * p : 2 * (v_tp + RPP * (p - KPASS))),
                                  kv_last);
                ids[p] = bt[BS16 ? j >> 4 : j / block_size];
            }
        };
        auto slot_of = [&](int j, int id) __attribute__((always_inline)) {
            const int phys = min(max(id, 0), max_phys);  // a bad block id stays in the pool
            return (uint32_t)(phys * block_size + (BS16 ? j & 15 : j % block_size));
        };
        // rows past the item's range read zeros
        auto load_step = [&](int kv0, const int* ids, u32x4* kd, u32x4 (*vd)[2]) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < KPASS; p++) {
                const int j = kv0 + k_row + RPP * p;
                const uint32_t o = slot_of(j, ids[p]) * ROW_BYTES + k_col * (uint32_t)sizeof(T);
                kd[p] = __builtin_amdgcn_raw_buffer_load_b128(k_rsrc, j < kv_end ? o : PT_OOR, 0, 0);
            }
#pragma unroll
            for (int p = 0; p < VPASS; p++) {
                const int j = kv0 + 2 * (v_tp + RPP * p);
                const uint32_t o = slot_of(j, ids[KPASS + p]) * ROW_BYTES + v_col * (uint32_t)sizeof(T);
#pragma unroll
                for (int t = 0; t < 2; t++)
                    vd[p][t] = __builtin_amdgcn_raw_buffer_load_b128(
                        v_rsrc, j + t < kv_end ? o + t * ROW_BYTES : PT_OOR, 0, 0);
            }
        };
        auto store_step = [&](int buf, const u32x4* kd, const u32x4 (*vd)[2]) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < KPASS; p++)
                *reinterpret_cast<u32x4*>(kt(buf) + (k_row + RPP * p) * KP + k_col) = kd[p];
#pragma unroll
            for (int p = 0; p < VPASS; p++) {
                uint16_t* dst = vt(buf) + v_col * VP + sigma16(2 * (v_tp + RPP * p));
#pragma unroll
                for (int e = 0; e < 8; e++) {  // V^T row v_col + e: the two tokens as one dword
                    const uint32_t a = vd[p][0][e >> 1], b = vd[p][1][e >> 1];
                    *reinterpret_cast<uint32_t*>(dst + e * VP) =
                        (e & 1) ? perm_hi16(a, b) : perm_lo16(a, b);
                }
            }
        };

        int ids[NID];
        u32x4 kd[KPASS], vd[VPASS][2];
        const int n_st = (kv_end + KT - 1) / KT;
        load_ids(0, ids);
        // Q^T as the B operand: lane (h2, r) holds row r, dims 16kk + 8h2 .. + 7
        u32x4 qb[NKQ];
        {
            const T* qp = q + (int64_t)(row0 + min(i, q_len - 1)) * q_st + (int64_t)head * q_sh + 8 * h2;
#pragma unroll
            for (int kk = 0; kk < NKQ; kk++) qb[kk] = *reinterpret_cast<const u32x4*>(qp + 16 * kk);
        }
        float m = -INFINITY, l = 0.0f;
        f32x16 o[NMT];
#pragma unroll
        for (int t = 0; t < NMT; t++)
#pragma unroll
            for (int e = 0; e < 16; e++) o[t][e] = 0.0f;
        if (n_st > 0) {
            load_step(0, ids, kd, vd);
            load_ids(KT, ids);
            __syncthreads();  // the last item's states are read
            store_step(0, kd, vd);
        }
        __syncthreads();
        for (int st = 0; st < n_st; st++) {
            const int buf = st & 1, kv0 = st * KT + 32 * ks;  // the wave's first position
            const bool more = st + 1 < n_st;
            if (more) {
                load_step((st + 1) * KT, ids, kd, vd);
                load_ids((st + 2) * KT, ids);
            }
            if (kv0 < w_end) {  // uniform over the wave
                // scores of the wave's tiles (every SPLIT-th 32 positions of the step); a tile past
                // the wave's range is zeros, masked like the rest
                f32x16 sc[SUB];
#pragma unroll
                for (int u = 0; u < SUB; u++) {
                    const uint16_t* kr = kt(buf) + (32 * (ks + SPLIT * u) + r) * KP + 8 * h2;
#pragma unroll
                    for (int e = 0; e < 16; e++) sc[u][e] = 0.0f;
#pragma unroll
                    for (int kk = 0; kk < NKQ; kk++)
                        sc[u] = mfma32x32x16<T>(*reinterpret_cast<const u32x4*>(kr + 16 * kk), qb[kk], sc[u]);
                }
                if (kv0 + 32 * SPLIT * (SUB - 1) + 31 > w_full) {  // the last tile crosses some row's limit
                    const int tl = lim - kv0 - 4 * h2;
#pragma unroll
                    for (int u = 0; u < SUB; u++)
#pragma unroll
                        for (int e = 0; e < 16; e++)
                            if (32 * SPLIT * u + 8 * (e >> 2) + (e & 3) > tl) sc[u][e] = -INFINITY;
                }
                float tm = sc[0][0];
#pragma unroll
                for (int u = 0; u < SUB; u++)
#pragma unroll
                    for (int e = 0; e < 16; e += 2) tm = vmax(vmax(tm, sc[u][e]), sc[u][e + 1]);
                tm = max_across_halves(tm) * scale_log2;  // scale > 0
                const float m_new = fmaxf(m, tm);
                const float nm = m_new == -INFINITY ? 0.0f : -m_new;  // nothing visible: all p = 0
                if (__builtin_amdgcn_ballot_w64(m_new > m) != 0) {
                    const float alpha = fast_exp2(m + nm);
                    l *= alpha;
#pragma unroll
                    for (int t = 0; t < NMT; t++) o[t] *= alpha;
                }
                m = m_new;
                float ps = 0.0f;
                const uint16_t* vr = vt(buf) + r * VP + 32 * ks + 8 * h2;
#pragma unroll
                for (int u = 0; u < SUB; u++)
#pragma unroll
                    for (int kk2 = 0; kk2 < 2; kk2++) {  // 16 tokens each
                        u32x4 ph, pl;
#pragma unroll
                        for (int y = 0; y < 4; y++) {
                            const float a = fast_exp2(fmaf(sc[u][8 * kk2 + 2 * y], scale_log2, nm));
                            const float b = fast_exp2(fmaf(sc[u][8 * kk2 + 2 * y + 1], scale_log2, nm));
                            const uint32_t hi = pack2<T>(a, b);
                            ph[y] = hi;
                            if constexpr (HILO) {
                                pl[y] = pack2<T>(a - lo_f32<T>(hi), b - hi_f32<T>(hi));
                                ps += a + b;
                            } else {  // the sum of the weights that enter the product
                                ps += lo_f32<T>(hi) + hi_f32<T>(hi);
                            }
                        }
#pragma unroll
                        for (int t = 0; t < NMT; t++) {
                            const u32x4 v = *reinterpret_cast<const u32x4*>(vr + 32 * t * VP + 32 * SPLIT * u + 16 * kk2);
                            o[t] = mfma32x32x16<T>(v, ph, o[t]);
                            if constexpr (HILO) o[t] = mfma32x32x16<T>(v, pl, o[t]);
                        }
                    }
                l += ps;
            }
            if (more) store_step(buf ^ 1, kd, vd);
            __syncthreads();
        }
        l = sum_across_halves(l);
        // fold the shares' states (the last step's barrier is behind every read of the tiles)
        float* st = reinterpret_cast<float*>(lds) + lane;
        auto state = [&](int share) { return st + ((share - 1) * SLOTS + wq) * NS * 64; };
        if (ks) {
            float* d = state(ks);
#pragma unroll
            for (int t = 0; t < NMT; t++)
#pragma unroll
                for (int e = 0; e < 16; e++) d[(16 * t + e) * 64] = o[t][e];
            d[16 * NMT * 64] = m;
            d[(16 * NMT + 1) * 64] = l;
        }
        __syncthreads();
        if (!ks && active && i < q_len) {
            float mm = m, f[SPLIT];
#pragma unroll
            for (int y = 1; y < SPLIT; y++) mm = fmaxf(mm, state(y)[16 * NMT * 64]);
            const float mz = mm == -INFINITY ? 0.0f : mm;
            f[0] = fast_exp2(m - mz);
            l *= f[0];
#pragma unroll
            for (int y = 1; y < SPLIT; y++) {
                f[y] = fast_exp2(state(y)[16 * NMT * 64] - mz);
                l += f[y] * state(y)[(16 * NMT + 1) * 64];
            }
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;  // no visible position: a zero row
            const int64_t obase = (int64_t)(row0 + i) * o_st + (int64_t)head * o_sh + 4 * h2;
#pragma unroll
            for (int t = 0; t < NMT; t++)
#pragma unroll
                for (int e = 0; e < 16; e += 4) {
                    float v[4];
#pragma unroll
                    for (int y = 0; y < 4; y++) {
                        float a = o[t][e + y] * f[0];
#pragma unroll
                        for (int z = 1; z < SPLIT; z++) a += state(z)[(16 * t + e + y) * 64] * f[z];
                        v[y] = a * inv;
                    }
                    store_run<4>(out, out_dtype, obase + 32 * t + 2 * e, v);
                }
        }
    }
}

// Items of a batch at `slots` slots an item, counted from its rows.
static int64_t thin_items(int slots, int num_seqs, int total_q, int num_heads, int n_rep) {
    const int hw = std::min(item_heads(n_rep), slots), rows = 32 * (slots / hw);
    return (int64_t)(num_heads / n_rep) * ((n_rep + hw - 1) / hw) * (total_q / rows + num_seqs);
}

static int g_prefill_small = 1;  // a test / tuning switch

// Slots per item of a small batch that runs here (varlen_prefill.hip's shape checks hold; `cus`: CUs
// of the device), 0 where varlen_prefill.hip takes it. Over a long cached prefix all items are alike,
// and a batch takes items per CU, rounded up, times ~12 ns a position with two slots and ~18 with
// four, where varlen_prefill.hip's larger items take ~20 and are fewer: two slots up to one item per
// CU, then four up to one, whatever the kv lengths. us there / here: 14 / 2 heads, 1 x 1,000 rows 29.6
// / 20.7, 1 x 2,000 51.2 / 44.4; 8 / 8 heads, 1 x 2,000 50.2 / 32.5; 32 / 32, 3 x U[64, 512] 17.6 /
// 13.3; 32 / 8, 4 x 191 behind 4,096 tokens 95 / 79; past that line 14 / 2, 16 x U[64, 286] behind
// 1,024 35 / 47. A single prompt without a prefix (by kv_cap) has items of every length, which the
// snake pairs: two slots up to one item per CU at four (1 x 2,000 rows 39.9 against 44.4 with four),
// four up to one and a half (1 x 2,867 rows 66.7 there, 58.8 here). Of 21,794 batches of 1-64
// sequences behind 0-4,096 tokens one is more than 3% slower than there (4%).
// At head_dim 128 the same kernel was even (32 / 8 heads, 1 x 1,000 rows 39.9 / 39.3, 3 x U[64, 512]
// 20.8 / 21.2; 1 x 2,000 74 / 79; only 1 x 256 gained, 17.0 / 15.6), with the step's wait as it is.
// kv_cap: a bound on the kv lengths (the positions that a row of the block table holds, or less).
int prefill_thin_slots(int num_seqs, int max_seqlen_q, int total_q, int64_t kv_cap, int num_heads,
                       int n_rep, int head_dim, int cus) {
    if (g_prefill_small == 0 || head_dim != PT_D || num_seqs > 64 || max_seqlen_q > 65536) return 0;
    if (g_prefill_small > 1) return g_prefill_small;
    if (thin_items(2, num_seqs, total_q, num_heads, n_rep) <= cus) return 2;
    const int64_t items = thin_items(4, num_seqs, total_q, num_heads, n_rep);
    if (num_seqs == 1 && kv_cap <= (int64_t)total_q + 256)
        return items <= cus ? 2 : items <= cus + cus / 2 ? 4 : 0;
    return items <= cus ? 4 : 0;
}

int launch_prefill_thin(int dtype, int out_dtype, void* out, int64_t o_st, int64_t o_sh,
                        const void* q, int64_t q_st, int64_t q_sh, const void* k_pool,
                        const void* v_pool, const int32_t* cu, const int32_t* q_rows,
                        const int32_t* kv_lens, const int32_t* bt, int max_blocks, int num_seqs,
                        int max_seqlen_q, int total_q, int num_heads, int n_rep, int block_size,
                        int64_t num_slots, float scale, int slots, int cus, bool persistent,
                        hipStream_t stream) {
    const int kv_heads = num_heads / n_rep;
    const int hw = std::min(item_heads(n_rep), slots), rows = 32 * (slots / hw);
    const int n_qt = (max_seqlen_q + rows - 1) / rows;
    const int64_t items = thin_items(slots, num_seqs, total_q, num_heads, n_rep);
    const int grid = (int)(persistent ? std::min<int64_t>(items, cus) : items);
    if (grid <= 0) return FLOUR_OK;
#define FLOUR_PT(T, B, S)                                                                       \
    prefill_thin_kernel<T, B, S><<<dim3(grid), dim3(PT_WAVES * 64), 0, stream>>>(                \
        out, out_dtype, o_st, o_sh, static_cast<const T*>(q), q_st, q_sh,                        \
        static_cast<const T*>(k_pool), static_cast<const T*>(v_pool), cu, q_rows, kv_lens, bt,   \
        max_blocks, num_seqs, kv_heads, n_rep, hw, block_size, num_slots, n_qt,                  \
        scale * 1.4426950408889634f)
#define FLOUR_PT_T(T)                           \
    do {                                        \
        if (block_size == 16 && slots == 4)     \
            FLOUR_PT(T, true, 4);               \
        else if (block_size == 16)              \
            FLOUR_PT(T, true, 2);               \
        else if (slots == 4)                    \
            FLOUR_PT(T, false, 4);              \
        else                                    \
            FLOUR_PT(T, false, 2);              \
    } while (0)
    if (dtype == FLOUR_DTYPE_BF16)
        FLOUR_PT_T(bf16_t);
    else
        FLOUR_PT_T(f16_t);
#undef FLOUR_PT_T
#undef FLOUR_PT
    return check_hip(hipGetLastError(), "varlen_prefill (small batch) launch");
}

}  // namespace flour

using namespace flour;

// 16-bit prefill at head_dim 64: 1 (the default): small batches on this kernel, by the rule above;
// 0: none; 2, 4: every batch of up to 64 sequences, with that many slots an item. A test / tuning
// switch.
extern "C" int flour_hip_set_prefill_small(int mode) {
    if (mode != 0 && mode != 1 && mode != 2 && mode != 4) {
        set_error("set_prefill_small: mode %d is not 0, 1, 2 or 4", mode);
        return FLOUR_ERR_INVALID_ARGUMENT;
    }
    g_prefill_small = mode;
    return FLOUR_OK;
}
