// Attention column means on gfx950 (MI355X): the kernels of the general two-pass path.  The column pass comes first.
// (Templates; fcs_stream_{rows,cols}.hip and fcs_stream_{rows,cols}_grouped.hip instantiate one pass each, so that the
// four compile side by side.)
//
// Given the row statistics of pass 1 (row maximum m_i and l_i = sum_j 2^((s_ij - m_i) * c),
// c = scale * log2(e)), this kernel adds up  p_ij = 2^((s_ij - m_i) * c - log2 l_i)  over heads and
// query rows for every key j.
//
// Orientation  S = Q_tile * K_tile^T  on v_mfma_f32_32x32x16: a lane owns ONE key (column
// lane % 32 of the tile) and 16 query rows of it in its accumulator registers.
//   * Q is the stationary operand: a wave keeps 32 * NB query rows of one head in registers.
//   * The per-row constant  n_i = -log2(l_i) / c  enters the matrix pipe as the INITIAL
//     accumulator value of the row, so the scores leave the MFMAs as  s_ij + n_i  and
//     p_ij = 2^(c * (s_ij + n_i))  costs one multiply and one v_exp_f32.  (Rows that pass 1 had
//     to stabilise, m_i != 0, are rare: a unit that holds one (FOLD: a wave) starts its
//     accumulators at 0, so that its scores carry the very bits pass 1 saw, subtracts m_i before
//     the scale and log2 l_i after it.)
//   * Summing p over the rows of a tile is in-lane; the two half-waves (which hold different
//     rows of the same keys) are added with v_permlane32_swap, and the wave adds its total for
//     the stage's keys into ITS OWN slice of an LDS accumulator (plain read-modify-write; a slot has
//     one writer, stage after stage, so the order of additions is fixed).
//   * K is streamed: the waves of a workgroup share 64-key stages that they fetch with
//     global_load_lds_dwordx4 straight into an LDS ring, several stages ahead, XOR-swizzled so
//     that the operand reads (ds_read_b128, 32 rows a row pitch apart) are conflict-free.  One
//     workgroup barrier per stage; the DMA is waited for by hand with s_waitcnt vmcnt(n).
//   * The stream has two loops: the stages that every row of a wave sees run in one without any test of position
//     (unrolled over the ring), the others (diagonal, last partial stage) in a short rolled one; stages that no row
//     of a wave sees cost it a barrier and its share of the fetch.  With the masked code inlined at every tile the
//     kernel was 2.3 times as long and needed 254 registers at D 128 (now 211).  Measured against that form, in
//     turn: B 1, H 32, Q 512, K 65536, D 128 607 -> 599 us per call, causal B 1, H 32, S 900, D 128 38.5 -> 34.7,
//     S 4096 bf16 233 -> 229.
//     In the rolled loop two chains come before their exponent work, so that the first tile's runs under the second
//     chain: two tiles of a key fragment for 64-row waves, the two fragments of the stage for 32-row waves, which also
//     read the next stage's first fragment ahead (not at D 256, where that was 1 .. 3 % slower).  It matters for decode windows, whose masked
//     stages lie in the last key split alone, whose workgroups end the launch.  Against one tile at a time: H 32, Q 128,
//     K 16384, D 128 on keys that change from call to call 83.8 -> 82.0 us (82.2 with the masked code inlined), H 8,
//     Q 512, K 4096, D 256 37.6 -> 34.4 (34.9).  Carrying the last tile over to the next stage, as the plain loop does,
//     was 0.1 % faster there and up to 7 % slower on short streams (H 8, Q 128, K 1000, D 64 16.3 -> 17.3 us); for
//     64-row waves it was slower throughout (H 32, S 2000, D 64 58.0 -> 59.8).
// A workgroup owns a chunk of keys (at most kColChunkMax, the LDS accumulator) and walks over a
// group of (head, row block) units, re-streaming its chunk for each; at the end the waves'
// slices are added in wave order and written as one partial slab (or the means directly, when
// there is a single group).  Causal alignment  j <= k_past + i  (reference:
// flash_colsum/kernel_causal.py:39,57,113): the stage loop stops at the last key any row of the
// unit sees, only stages on the diagonal (or past the last key) take the masked code path.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fcs_device.h"
#include "fcs_kernels.h"

namespace fcs {

namespace {

#define FCS_WAIT_VM(N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory")
#define FCS_WAIT_LGKM0() asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory")

// 64 lanes x 16 bytes from global memory straight into LDS: lane L's piece lands at dst + 16 * L
// (dst is wave-uniform)
__device__ __forceinline__ void dma16(const char *src, char *dst)
{
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src,
                                     (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
}

// workgroup barrier that also orders this wave's LDS accesses around it (the bare s_barrier
// intrinsic is neither a fence for the compiler nor a wait for outstanding LDS writes)
__device__ __forceinline__ void block_sync() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void block_barrier() { asm volatile("s_barrier" ::: "memory"); }

__device__ __forceinline__ uint32_t lds_addr(const void *p)
{
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char *)p;
}

// position swizzle of the 16-byte pieces of a stage row: rows a row pitch apart must not share banks
template <int D>
__device__ __forceinline__ int row_swizzle(int row)
{
    return D == 64 ? ((row >> 1) & 7) : (row & 15);
}

// source of the 16-byte pieces that lie past the tensor's head dim (kernels compiled for a wider head)
__device__ unsigned int g_zero_piece[4];

// FOLD: the rows of a unit are those of ALL query heads that share a key head, laid end to end: row v of key head hk
// is row v % q_rows of query head hk * fold + v / q_rows.  v / q_rows through a multiply-high; fold_magic is
// ceil(2^31 / q_rows), exact while v * q_rows < 2^31 (checked by the plan).
__device__ __forceinline__ int fold_head(int v, uint32_t magic) { return (int)__umulhi((uint32_t)v << 1, magic); }

// this lane's averaged row v (clamped to the last one): its first element in Q
template <bool FOLD>
__device__ __forceinline__ const _Float16 *q_row_ptr(const Args &a, int b, int h, int v)
{
    if constexpr (FOLD) {
        v = min(v, a.v_rows - 1);
        const int gi = fold_head(v, a.fold_magic);
        return a.q + (int64_t)b * a.qs_b + (int64_t)(h * a.fold + gi) * a.qs_h + (int64_t)(v - gi * a.q_rows) * a.qs_s;
    } else {
        return a.q + (int64_t)b * a.qs_b + (int64_t)h * a.qs_h + (int64_t)min(v, a.Sq - 1) * a.qs_s;
    }
}

// causal calls: one past the last row (within its head) of the rows [v0, v1) that see the most keys, and the row that
// sees the fewest of the wave's `n` rows from v on
template <bool FOLD>
__device__ __forceinline__ int rows_past(const Args &a, int v1)
{
    return FOLD ? a.q_rows : min(v1, a.q_rows);
}
template <bool FOLD>
__device__ __forceinline__ int rows_first(const Args &a, int v, int n)
{
    if constexpr (FOLD) {
        const int gi = fold_head(v, a.fold_magic);
        return (v + n <= (gi + 1) * a.q_rows) ? v - gi * a.q_rows : 0;
    } else {
        return v;
    }
}

// Masked work on a fragment of 32 rows from row v0 on (wave-uniform): add(ahead) with ahead(i) = the rows of the heads
// before the row of accumulator register i, which `rel` has to be raised by.  Folded rows: a fragment inside one head, the
// usual case, raises `rel` once; only one that holds rows of several heads divides per register.
template <bool FOLD, class F>
__device__ __forceinline__ void mask_rows(const Args &a, int v0, int g4, int &rel, F add)
{
    if constexpr (FOLD) {
        const int h0 = fold_head(v0, a.fold_magic);
        if (h0 == fold_head(v0 + 31, a.fold_magic)) {
            rel += h0 * a.q_rows;
            add([](int) { return 0; });
        } else {
            int v = v0 + g4;
            asm volatile("" : "+v"(v));  // formed here, not kept for every register through the stream
            add([&](int i) { return fold_head(v + 8 * (i >> 2) + (i & 3), a.fold_magic) * a.q_rows; });
        }
    } else {
        add([](int) { return 0; });
    }
}

// How many of the nst stages from key k0 on lie within the keys up to `thr`, which all rows of a wave see
__device__ __forceinline__ int plain_stages(int k0, int nst, int thr)
{
    return (thr + 1 >= k0) ? min(nst, (thr + 1 - k0) / kStageKeys) : 0;
}

// ... and how many of them hold a key up to `thr`, the last one that any row of it sees
__device__ __forceinline__ int seen_stages(int k0, int nst, int thr)
{
    return (thr >= k0) ? min(nst, (thr - k0) / kStageKeys + 1) : 0;
}

// Rows beyond the unstabilised range: rows laid end to end (FOLD) are stabilised head by head, the waves that hold such a head;
// others with their whole block.  (PRE: the block too, since a unit with stabilised rows takes the raw operand throughout.)
// Error against 64 bits of a call with such rows, as without folding (16 on 2 heads, Q 128, K 65536, D 64: 9.2e-7 and 9.1e-7).
template <bool PRE, bool FOLD>
constexpr bool kRedoHeads = FOLD && !PRE;

// column pass: how the exponent is taken
constexpr int kFormRaw = 0, kFormPrescaled = 1, kFormShifted = 2;

// ceiling of a row's sum of exponentials in the pre-scaled variants: keeps every score of the common path
// below 20 in the exponent's unit, which bounds what rounding Q * c to fp16 can do to it (the error of a
// score grows with the spread of the scores; peaked rows, whose few large probabilities are not averaged
// with thousands of others, are the ones this sends to the exact sweeps)
constexpr float kRowSumHiPre = 1048576.f;  // 2^20

// Pre-scaled stationary operand: q * cs in fp32, rounded to fp16 (cs = c with the scale's sign).  The
// scores then leave the matrix pipe in the exponent's unit and the per-score multiply disappears.  Both
// passes form the operand with this one function, so they see the same score bits.
__device__ __forceinline__ half8 prescale(half8 v, float cs)
{
    half8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = (_Float16)((float)v[e] * cs);
    return r;
}

}  // namespace

// PRE (fp16, D = 64; chosen by the launcher when at least 16384 (head, row) pairs are averaged and
// |scale| <= 1/8): for the keys below a.pre_end the stationary operand is Q * c rounded to fp16, the row constant
// is -log2 l_i, and p_ij = 2^(s'_ij - log2 l_i) costs a v_exp_f32 alone.  Pass 1 made l_i from the same scores:
// both passes decide per 64-key stage, by the stage's position alone (stages that end at or below a.pre_end, a
// multiple of 64: every key of a non-causal call; the keys that EVERY row sees of a causal one, whose last keys
// are averaged over few rows and keep the raw operand).  A unit therefore streams in up to two phases, the
// pre-scaled stages first, then the raw ones after reloading Q.  Units with a stabilised row keep the raw operand
// and the two-constant form throughout.
template <int D, int NB, int WAVES, bool BF, bool PRE, bool FOLD>
__global__ __launch_bounds__(64 * WAVES, 2) void fcs_colstream_kernel(const Args a)
{
    static_assert(!PRE || (!BF && D == 64), "the pre-scaled variant exists for fp16 operands and 64-wide heads");
    constexpr int THREADS = 64 * WAVES;
    constexpr int NT = D / 16;                 // MFMA steps along the head dim
    constexpr int NTA = NT < 8 ? NT : 8;       // operand addresses: the swizzle stays below piece 16, step t + 8 is 256 bytes on
    constexpr int KT = kStageKeys;             // 64 keys per stage
    constexpr int NA = KT / 32;                // key fragments per stage
    constexpr int ROWS_W = 32 * NB;            // query rows per wave
    constexpr int BLOCK_ROWS = WAVES * ROWS_W;
    constexpr int ROW_BYTES = D * 2;
    constexpr int PPR = D / 8;                 // 16-byte pieces per row
    constexpr int STAGE_BYTES = KT * ROW_BYTES;
    constexpr int IPW = KT * PPR / THREADS;    // DMA instructions per wave per stage
    constexpr int NS = col_ring_slots(D, WAVES);
    constexpr int CHUNK = col_chunk_max(D, WAVES);
    static_assert(IPW >= 1 && KT * PPR == IPW * THREADS, "a stage is a whole number of DMA instructions per wave");
    static_assert(NS >= 3, "the ring holds the stage in use, the next one and at least one in flight");
    __shared__ __attribute__((aligned(16))) char ring[NS * STAGE_BYTES];
    __shared__ __attribute__((aligned(16))) float colw[WAVES * CHUNK];  // per-wave column sums of the chunk
    __shared__ __attribute__((aligned(16))) float nl_s[BLOCK_ROWS];     // per-row constants of the current unit: -log2(l_i) / c
    __shared__ __attribute__((aligned(16))) float np_s[PRE ? BLOCK_ROWS : 4];  // the same for pre-scaled scores: -log2(l_i)
    __shared__ __attribute__((aligned(16))) float lg_s[BLOCK_ROWS];     // log2 l_i, used by units with stabilised rows
    __shared__ __attribute__((aligned(16))) float cm_s[BLOCK_ROWS];     // -m_i of those units
    __shared__ int shift_s[WAVES];                                       // per wave: one of its rows is stabilised

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int cx, grp, b;  // chunks of one (group, batch entry) stream the same Q: neighbours in launch order
    xcd_contiguous_block((int)blockIdx.x, a.c_nchunks, a.c_groups, a.B, cx, grp, b);  // a one-dimensional grid: no axis limit
    const int c0 = cx * a.c_chunk;                     // first key of the chunk
    const int c1 = min(a.Sk, c0 + a.c_chunk);          // one past its last key
    const int u_begin = grp * a.c_upg, u_end = min(a.v_heads * a.c_nrb, u_begin + a.c_upg);
    const float cmul = (a.c == 0.f) ? 1.f : a.c;       // scale 0: Q is zeroed instead and n_i = -log2 l_i

    // ---- this wave's slice of the column accumulator
    float *colw_w = colw + wave * CHUNK;
    for (int i = lane * 4; i < CHUNK; i += 256) *reinterpret_cast<floatx4 *>(colw_w + i) = floatx4{0.f, 0.f, 0.f, 0.f};

    // ---- DMA geometry: piece P of a stage goes to LDS byte 16 * P; it is piece pos ^ swizzle(row)
    // of stage row `row`, so that row r keeps piece p at position p ^ swizzle(r)
    uint32_t g_off[IPW];   // byte offset of this lane's piece from the stage's first key row (dense stage)
#pragma unroll
    for (int j = 0; j < IPW; ++j) {
        const int P = (wave * IPW + j) * 64 + lane;
        const int row = P / PPR, pos = P % PPR;
        g_off[j] = (uint32_t)row * (uint32_t)(a.ks_s * 2) + (uint32_t)((pos ^ row_swizzle<D>(row)) * 16);
    }
    char *ring_w = ring + wave * (IPW * 1024);  // where this wave's pieces of a stage land inside a slot
    // operand read-back: lane (n, g) takes, for MFMA step t, piece 2t + g of row n (+ 32 per key fragment)
    uint32_t take[NTA];
#pragma unroll
    for (int t = 0; t < NTA; ++t)
        take[t] = lds_addr(ring) + (uint32_t)(n * ROW_BYTES + (((2 * t + g) ^ row_swizzle<D>(n)) * 16));

    for (int u = u_begin; u < u_end; ++u) {
        const int h = u / a.c_nrb, rb = u - h * a.c_nrb;
        const int row0 = rb * BLOCK_ROWS;                        // first query row of the unit
        // keys of the chunk that some row of the unit sees
        int kend = c1;
        if (a.causal) kend = min(kend, a.k_past + rows_past<FOLD>(a, row0 + BLOCK_ROWS));
        const int nst = (kend > c0) ? (kend - c0 + KT - 1) / KT : 0;
        if (nst == 0) continue;  // block-uniform

        // ---- per-row constants, merged over the key splits of pass 1
        {
            const int qi = row0 + tid;
            float nl = -INFINITY;  // a row that is not averaged: every p comes out as 2^-inf = 0
            float mm = 0.f, lg = 0.f;
            if (tid < BLOCK_ROWS && qi < a.v_rows) {
                const int64_t bh = (int64_t)b * a.v_heads + h;
                if (a.n_chunks == 1) {
                    const float2 v = a.lse[bh * a.rows_pad + qi];
                    mm = v.x;
                    lg = v.y;
                } else {
                    const float2 *p = a.ml + bh * a.n_chunks * a.rows_pad + qi;
                    mm = kNegBig * 4.f;
                    float ll = 0.f;
                    for (int ch0 = 0; ch0 < a.n_chunks; ch0 += 8) {  // eight loads in flight; folded in split order
                        float2 v[8];
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            v[j].x = kNegBig * 4.f;
                            v[j].y = 0.f;
                            if (ch0 + j < a.n_chunks) v[j] = p[(int64_t)(ch0 + j) * a.rows_pad];
                        }
#pragma unroll
                        for (int j = 0; j < 8; ++j) {  // fixed order: bit-reproducible
                            // A split that pass 1 left unstabilised reports m = 0 and a sum of up to 2^110;
                            // next to a stabilised split its weight 2^((0 - m) * c) alone underflows although
                            // the product does not: the weights are applied as two square roots.
                            const float mn = fmaxf(mm, v[j].x);
                            const float wa = fast_exp2((mm - mn) * (0.5f * a.c)), wb = fast_exp2((v[j].x - mn) * (0.5f * a.c));
                            ll = (ll * wa) * wa + (v[j].y * wb) * wb;
                            mm = mn;
                        }
                    }
                    lg = fast_log2(ll);
                }
                nl = (a.c == 0.f) ? -lg : -lg / a.c;
            }
            // a stabilised row switches the whole unit, or its wave (kRedoHeads), to the two-constant form
            const bool sh = __builtin_amdgcn_ballot_w64(mm != 0.f) != 0;
            if (lane == 0) shift_s[wave] = sh ? 1 : 0;
            if (tid < BLOCK_ROWS) {
                nl_s[tid] = nl;
                if (PRE) np_s[tid] = (nl == -INFINITY) ? -INFINITY : -lg;
                lg_s[tid] = lg;
                cm_s[tid] = (nl == -INFINITY) ? -INFINITY : -mm;
            }
        }

        // ---- stationary operand: this wave's query rows of head h, as they are in memory
        const int qw0 = row0 + wave * ROWS_W;
        half8 qf[NB][NT];
        auto load_q_rows = [&]() {
            int lane_o = lane;
            asm volatile("" : "+v"(lane_o));  // addresses are formed here, not kept for a second call
            const int n_o = lane_o & 31, g_o = lane_o >> 5;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const _Float16 *row = q_row_ptr<FOLD>(a, b, h, qw0 + nb * 32 + n_o) + g_o * 8;
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    half8 v = kZero8;  // channels past the tensor's head dim are zeros
                    if (t * 16 + g_o * 8 < a.D) v = load8(row + t * 16);
                    if (a.c == 0.f) v = kZero8;
                    qf[nb][t] = v;
                }
            }
        };
        // the form the matrix pipe takes: pre-scaled (sign included), or raw with the scale's sign
        auto shape_q = [&](bool scaled) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    if (PRE && scaled) qf[nb][t] = prescale(qf[nb][t], a.negate ? -a.c : a.c);
                    else if (a.negate) qf[nb][t] = flip_sign(qf[nb][t]);
                }
        };
        load_q_rows();
        const char *kp = reinterpret_cast<const char *>(a.k + (int64_t)b * a.ks_b +
                                                        (int64_t)kv_head(h, a.kv_group, a.kv_magic) * a.ks_h);
        const int64_t k_row_b = a.ks_s * 2;

        // stage `st` of the unit into ring slot `slot` (stages past the last one repeat it, so that the
        // number of DMA instructions in flight at every wait is a compile-time constant).
        auto fetch_stage = [&](int st, int slot) {
            const int kb = c0 + min(st, nst - 1) * KT;
            char *dst = ring_w + slot * STAGE_BYTES;
            // whole stage inside the tensor, rows as wide as compiled (wave-uniform; the other case out of line)
            if (__builtin_expect(kb + KT <= a.Sk && a.D == D, 1)) {
                const char *src = kp + (int64_t)kb * k_row_b;
#pragma unroll
                for (int j = 0; j < IPW; ++j) dma16(src + g_off[j], dst + j * 1024);
            } else {  // rows past the last key re-read it; the consumer masks them
                int lane_o = lane;
                asm volatile("" : "+v"(lane_o));  // formed here, not kept in registers through the stream
#pragma unroll
                for (int j = 0; j < IPW; ++j) {
                    const int P = (wave * IPW + j) * 64 + lane_o;
                    const int row = P / PPR, pos = P % PPR;
                    const int piece = pos ^ row_swizzle<D>(row);
                    const char *src = kp + (int64_t)min(kb + row, a.Sk - 1) * k_row_b + piece * 16;
                    if (piece * 8 >= a.D) src = reinterpret_cast<const char *>(g_zero_piece);  // past the head dim: zeros
                    dma16(src, dst + j * 1024);
                }
            }
        };

        // key fragment `na` of the stage in `slot` as MFMA B operand.  Inline assembly: the compiler
        // would make an ordinary LDS read wait for ALL outstanding DMA (vmcnt(0)).
        // The byte offset of (slot, fragment) is an immediate of the instruction: the stage loop
        // below is unrolled over the ring so that every slot number is a compile-time constant.
        auto take_frag = [&](auto off_c, half8 (&kf)[NT]) {
            constexpr int OFF = decltype(off_c)::value;
            constexpr int IMM = (OFF < 65536 - 256) ? OFF : 0;  // the offset field holds 16 bits
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const uint32_t ad = take[t % NTA] + (uint32_t)(OFF - IMM);
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(kf[t]) : "v"(ad), "n"(IMM + t / NTA * 256) : "memory");
            }
        };
        auto take_frag_at = [&](int off, half8 (&kf)[NT]) {  // the same at a run-time offset into the ring
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const uint32_t ad = take[t % NTA] + (uint32_t)off;
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(kf[t]) : "v"(ad), "n"(t / NTA * 256) : "memory");
            }
        };
        auto frag_wait = [&](half8 (&kf)[NT]) {
            if constexpr (NT == 4)
                asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(kf[0]), "+v"(kf[1]), "+v"(kf[2]), "+v"(kf[3])::"memory");
            else {
#pragma unroll
                for (int t0 = 0; t0 < NT; t0 += 8)
                    asm volatile("s_waitcnt lgkmcnt(0)"
                                 : "+v"(kf[t0]), "+v"(kf[t0 + 1]), "+v"(kf[t0 + 2]), "+v"(kf[t0 + 3]), "+v"(kf[t0 + 4]),
                                   "+v"(kf[t0 + 5]), "+v"(kf[t0 + 6]), "+v"(kf[t0 + 7])::"memory");
            }
        };

        // ---- prologue of the unit's first phase: NS - 1 stages in flight; stages 0 and 1 must have landed
        // before the first barrier
#pragma unroll
        for (int st = 0; st < NS - 1; ++st) fetch_stage(st, st);
        FCS_WAIT_VM((NS - 3) * IPW);
        block_sync();  // also publishes nl_s

        // The two-constant form: some row of the unit was stabilised by pass 1 (block-uniform), or, where pass 1 redoes single
        // heads, some row of this wave's (the flag of 64 rows: of two waves of 32).
        bool shifted = false;
        {
            int f = 0;
            const uint32_t ad = lds_addr(shift_s) + (uint32_t)((kRedoHeads<PRE, FOLD> ? wave * ROWS_W / 64 : lane % WAVES) * 4);
            asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(f) : "v"(ad) : "memory");
            shifted = __builtin_amdgcn_ballot_w64(f != 0) != 0;
        }
        // leading stages of the unit that run on the pre-scaled operand (block-uniform)
        const int n_pre = (!PRE || shifted) ? 0 : min(nst, max(0, (a.pre_end - c0) / KT));

        // rows of this wave relative to the causal diagonal; non-causal: every key below Sk is visible
        const int kp_eff = a.causal ? a.k_past : 0x3fffffff - a.Sq;
        const int thr_wave_min = a.causal ? min(a.k_past + rows_first<FOLD>(a, qw0, ROWS_W), a.Sk - 1) : a.Sk - 1;   // last key EVERY row of the wave sees
        const int thr_wave_max = a.causal ? a.k_past + (FOLD ? a.q_rows : qw0 + ROWS_W) - 1 : a.Sk - 1;             // last key ANY row of it sees
        // leading stages that every row of the wave sees: they run in the plain stream below
        const int n_plain = plain_stages(c0, nst, thr_wave_min);
        const int n_seen = seen_stages(c0, nst, thr_wave_max);  // those that some row of it sees

        // One phase: the stages [s0, s1) of the unit in one FORM: raw operand, pre-scaled operand, or the
        // two-constant form of a unit with a stabilised row.  `fetched`: the phase's first NS - 1 stages are already
        // in the ring (the unit's prologue above).
        auto run_phase = [&](auto form_c, const int s0, const int s1, const bool fetched) {
            constexpr int FORM = decltype(form_c)::value;
            constexpr bool SC = FORM == kFormPrescaled, SHIFTED = FORM == kFormShifted;
            if (!fetched) {
#pragma unroll
                for (int st = 0; st < NS - 1; ++st) fetch_stage(s0 + st, st);
                FCS_WAIT_VM((NS - 3) * IPW);
                block_sync();
            }
            floatx16 cinit[NB];  // row constants in accumulator layout: register i <-> row 8*(i/4) + 4*g + i%4
            int g_c = g;
            asm volatile("" : "+v"(g_c));  // addresses are formed here, not kept from unit to unit
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    floatx4 v = {0.f, 0.f, 0.f, 0.f};
                    if (!SHIFTED) {  // inline assembly for the same reason as the operand reads
                        const uint32_t ad = lds_addr(SC ? np_s : nl_s) + (uint32_t)((wave * ROWS_W + nb * 32 + 8 * i4 + 4 * g_c) * 4);
                        asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(ad) : "memory");
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) cinit[nb][4 * i4 + j] = v[j];
                }

            // A stage is NA * NB tiles of 32 rows x 32 keys; tile q = na * NB + nb uses key fragment na and
            // accumulator q & 1.
            constexpr int TILES = NA * NB;
            static_assert(TILES % 2 == 0, "two accumulators alternate");
            static_assert(NA == 2, "fragment offsets below");
            half8 kf[NT];
            float cp[4] = {0.f, 0.f, 0.f, 0.f};  // running column sums of the fragment being exponentiated

            // Exponent work of one finished tile (kb_t: first key of its stage):
            //   drain_begin   requests the fragment's accumulator slot (first row fragment only)
            //   drain_plain   every row sees every key of the tile
            //   drain_masked  tiles on the diagonal or past the last key
            //   drain_end     after the last row fragment: fold the half-waves, add into the wave's slice
            float col_old = 0.f;
            uint32_t col_ad = 0;
            auto drain_begin = [&](int kb_t, int na, int nb) {
                if (nb == 0) {
                    col_ad = lds_addr(colw_w) + (uint32_t)((kb_t - c0 + na * 32 + n) * 4);
                    asm volatile("ds_read_b32 %0, %1" : "=v"(col_old) : "v"(col_ad) : "memory");
                }
            };
            // two-constant form (rare): the accumulators started at 0, so the scores carry the very bits pass 1 saw;
            // m_i is subtracted before the scale and log2 l_i after it
            auto shifted_p = [&](const floatx16 &sc, int nb, int i4, float (&pr)[4]) {
                floatx4 l4, m4;
                int g_o = g;
                asm volatile("" : "+v"(g_o));  // addresses are formed here, not kept through the stream
                const uint32_t ro = (uint32_t)((wave * ROWS_W + nb * 32 + 8 * i4 + 4 * g_o) * 4);
                const uint32_t ad = lds_addr(lg_s) + ro, am = lds_addr(cm_s) + ro;
                asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                             : "=&v"(l4), "=&v"(m4)
                             : "v"(ad), "v"(am)
                             : "memory");
#pragma unroll
                for (int j = 0; j < 4; ++j) pr[j] = fast_exp2(fmaf(sc[4 * i4 + j] + m4[j], cmul, -l4[j]));
            };
            auto drain_plain = [&](const floatx16 &sc, int nb) {
                if constexpr (SHIFTED) {
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        float pr[4];
                        shifted_p(sc, nb, i4, pr);
#pragma unroll
                        for (int j = 0; j < 4; ++j) cp[j] += pr[j];
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 16; ++i) cp[i & 3] += fast_exp2(SC ? sc[i] : sc[i] * cmul);
                }
            };
            auto drain_masked = [&](const floatx16 &sc, int kb_t, int na, int nb) {
                const int key = kb_t + na * 32 + n;
                // visible  <=>  key < Sk  and  key - k_past - (row of register i) <= 0
                int rel = (key < a.Sk) ? key - kp_eff - (qw0 + 4 * g) : 0x3fffffff;
                asm volatile("" : "+v"(rel));
                auto add = [&](auto ahead) {  // ahead(i): rows of the heads before the row of register i (FOLD)
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        float pr[4];
                        if constexpr (SHIFTED) {
                            shifted_p(sc, nb, i4, pr);
                        } else {
#pragma unroll
                            for (int j = 0; j < 4; ++j) pr[j] = fast_exp2(SC ? sc[4 * i4 + j] : sc[4 * i4 + j] * cmul);
                        }
#pragma unroll
                        for (int j = 0; j < 4; ++j) cp[j] += (rel + ahead(4 * i4 + j) <= nb * 32 + 8 * i4 + j) ? pr[j] : 0.f;
                    }
                };
                mask_rows<FOLD>(a, qw0 + nb * 32, 4 * g, rel, add);
            };
            auto drain_end = [&](int nb) {
                if (nb == NB - 1) {
                    float tot = (cp[0] + cp[1]) + (cp[2] + cp[3]);
                    cp[0] = cp[1] = cp[2] = cp[3] = 0.f;
                    // v_permlane32_swap exchanges the upper half of its first operand with the lower half of
                    // its second: started from two copies of the value, one register then holds the lower
                    // half-wave's values in both halves and the other the upper half-wave's, so their sum is
                    // the total of the two half-waves in every lane.  (Inline assembly: given the same value
                    // twice, the builtin's two results were folded into one.)
                    float x = tot, y = tot;
                    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
                    tot = x + y;
                    // plain read-modify-write of the wave's own slot (LDS float atomics are slow): the old
                    // value was requested before the exponent work; both half-waves store the same total
                    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(col_old)::"memory");
                    tot += col_old;
                    asm volatile("ds_write_b32 %0, %1" ::"v"(col_ad), "v"(tot) : "memory");
                }
            };

            // MFMA chain of one tile alone
            auto chain = [&](int nb) {
                floatx16 c = mfma16<BF>(qf[nb][0], kf[0], cinit[nb]);
#pragma unroll
                for (int t = 1; t < NT; ++t) c = mfma16<BF>(qf[nb][t], kf[t], c);
                return c;
            };

            // ---- the plain stream: stages [s0, sp).  Software pipeline inside the wave: the MFMA chain of tile q is
            // issued BEFORE the exponent work of tile q - 1, so the matrix pipe and the VALU run together whatever
            // the phase of the other wave on the SIMD.  (Measured slower: the exponent work woven between the
            // chain's MFMAs, and the two waves of a SIMD in opposite order.)  Nothing in here depends on where the
            // stage lies; the waves of a block may leave it at different stages, since both loops pass one barrier
            // and issue the same fetches per stage.
            const int sp = min(s1, max(s0, n_plain));
            if (sp > s0) {
                take_frag(std::integral_constant<int, 0>{}, kf);
                floatx16 acc[2];
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.f;
                // one stage, in ring slot SLOT (compile-time; the phase's first stage is in slot 0)
                auto stage = [&](int st, auto slot_c) {
                    constexpr int SLOT = decltype(slot_c)::value;
                    const int kb = c0 + st * KT;
                    const bool first = SLOT == 0 && st == s0;
                    if (!first) {
                        // stage st + 1 has landed (this wave's pieces; the barrier extends that to everyone's), and
                        // every wave is done reading stage st - 1, whose slot takes the next fetch
                        FCS_WAIT_VM((NS - 3) * IPW);
                        block_barrier();
                    }
                    fetch_stage(st + NS - 1, (SLOT + NS - 1) % NS);
#pragma unroll
                    for (int q = 0; q < TILES; ++q) {
                        const int na = q / NB, nb = q % NB;
                        if (nb == 0) frag_wait(kf);
                        acc[q & 1] = chain(nb);
                        asm volatile("" : "+v"(acc[0]), "+v"(acc[1]));  // the chain stays where it was written
                        if (nb == NB - 1) {  // this fragment's last chain has been issued: read back the next one
                            if (na == 0) take_frag(std::integral_constant<int, SLOT * STAGE_BYTES + 32 * ROW_BYTES>{}, kf);
                            else take_frag(std::integral_constant<int, ((SLOT + 1) % NS) * STAGE_BYTES>{}, kf);
                        }
                        // the tile before: in this stage, or the last one of the previous stage
                        const int p_kb = (q > 0) ? kb : kb - KT;
                        const int p_na = (q > 0) ? (q - 1) / NB : NA - 1, p_nb = (q > 0) ? (q - 1) % NB : NB - 1;
                        if (q > 0 || !first) {
                            drain_begin(p_kb, p_na, p_nb);
                            drain_plain(acc[(q + 1) & 1], p_nb);
                            drain_end(p_nb);
                            asm volatile("" : "+v"(acc[0]), "+v"(acc[1]));
                        }
                    }
                };
                for (int st0 = s0; st0 < sp; st0 += NS) {
                    stage(st0, std::integral_constant<int, 0>{});
                    if (st0 + 1 < sp) stage(st0 + 1, std::integral_constant<int, 1>{});
                    if (st0 + 2 < sp) stage(st0 + 2, std::integral_constant<int, 2>{});
                    if (NS > 3 && st0 + 3 < sp) stage(st0 + 3, std::integral_constant<int, 3 % NS>{});
                }
                static_assert(NS <= 4, "unrolled above");
                frag_wait(kf);  // (the first fragment of the next stage, if there is one)
                drain_begin(c0 + (sp - 1) * KT, NA - 1, NB - 1);
                drain_plain(acc[(TILES - 1) & 1], NB - 1);
                drain_end(NB - 1);
            }

            // ---- the rest of the phase, in rolled loops (the ring slot is a run-time value): the stages on the diagonal or
            // past the last key as far as some row of the wave sees them, [sp, sv), then those that none of its rows sees
            const int sv = min(s1, max(sp, n_seen));
            int slot = (sp - s0) % NS;
            auto enter_stage = [&](int st) {
                if (st > s0) {
                    FCS_WAIT_VM((NS - 3) * IPW);
                    block_barrier();
                }
                fetch_stage(st + NS - 1, (slot == 0) ? NS - 1 : slot - 1);
                slot = (slot + 1 == NS) ? 0 : slot + 1;
            };
            auto drain_one = [&](const floatx16 &sc, int kb_t, int na, int nb) {
                drain_begin(kb_t, na, nb);
                drain_masked(sc, kb_t, na, nb);
                drain_end(nb);
            };
            if constexpr (NB == 1 && D <= 128) {
                if (sv > sp) {
                    floatx16 acc[2];
                    acc[0] = acc[1] = cinit[0];
                    if (sp == s0) take_frag(std::integral_constant<int, 0>{}, kf);  // else the plain stream has read it
                    frag_wait(kf);
#pragma unroll 1
                    for (int st = sp; st < sv; ++st) {
                        const int kb = c0 + st * KT, here = slot * STAGE_BYTES;
                        enter_stage(st);
                        frag_wait(kf);
                        acc[0] = chain(0);
                        asm volatile("" : "+v"(acc[0]), "+v"(acc[1]));
                        take_frag_at(here + 32 * ROW_BYTES, kf);
                        frag_wait(kf);
                        acc[1] = chain(0);
                        asm volatile("" : "+v"(acc[0]), "+v"(acc[1]));
                        take_frag_at(slot * STAGE_BYTES, kf);
                        drain_one(acc[0], kb, 0, 0);
                        drain_one(acc[1], kb, 1, 0);
                    }
                    frag_wait(kf);  // the read-back past the last stage is not used
                }
            } else {
                for (int st = sp; st < sv; ++st) {
                    const int kb = c0 + st * KT, here = slot * STAGE_BYTES;
                    enter_stage(st);
#pragma unroll 1
                    for (int s = 0; s < TILES / 2; ++s) {
                        floatx16 acc[2];
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            if (NB == 1 || q == 0) {
                                take_frag_at(here + (NB == 1 ? q : s) * 32 * ROW_BYTES, kf);
                                frag_wait(kf);
                            }
                            acc[q] = chain(NB == 1 ? 0 : q);
                        }
#pragma unroll
                        for (int q = 0; q < 2; ++q) drain_one(acc[q], kb, NB == 1 ? q : s, NB == 1 ? 0 : q);
                    }
                }
            }
            for (int st = sv; st < s1; ++st) enter_stage(st);
            // the look-ahead fetches issued past the last stage must be over before the ring (and nl_s) is reused by
            // the next phase or unit
            FCS_WAIT_VM(0);
            block_sync();
        };

        // (one call site per form, so that the code of each exists once)
        int raw0 = 0;  // first stage of the raw phase
        if (PRE && n_pre > 0) {
            shape_q(true);
            run_phase(std::integral_constant<int, kFormPrescaled>{}, 0, n_pre, true);
            raw0 = n_pre;
            if (raw0 < nst) load_q_rows();  // the unit's last stages (causal: keys that not every row sees)
        }
        if (raw0 < nst) {
            shape_q(false);
            if (shifted) run_phase(std::integral_constant<int, kFormShifted>{}, 0, nst, true);
            else run_phase(std::integral_constant<int, kFormRaw>{}, raw0, nst, raw0 == 0);
        }
    }

    // ---- add the waves' slices in wave order and store
    block_sync();
    const bool direct = (a.c_groups == 1);
    for (int i = tid; i < c1 - c0; i += THREADS) {
        float v = colw[i];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) v += colw[w * CHUNK + i];
        const int64_t o = (int64_t)b * a.Sk + c0 + i;
        if (direct) {
            a.out[o] = v * a.inv_norm;
            if (a.out_h) a.out_h[o] = (_Float16)(v * a.inv_norm);
        } else {
            a.partial[(int64_t)grp * a.B * a.Sk + o] = v;
        }
    }
}

// ------------------------------------------------------------------------------------
// pass 1 on the same machinery: row maximum and sum of exponentials of one (row block, head, key split)
// ------------------------------------------------------------------------------------
// Same orientation and stream as the column pass (Q stationary, K through the LDS-DMA ring), but the
// exponentials are added up per ROW: register i of a lane keeps the running sum of its row over the
// lane's keys for the whole split, and the 32 key lanes are added once at the end through LDS.
// Common case: 2^(c * s) without max subtraction, exact while every row sum of the split stays inside
// [2^-80, 2^110); a block that leaves that range redoes its keys in two more sweeps (row maxima, then
// sums of 2^((s - m) * c), the maximum subtracted before the scale).  FOLD: only the waves that hold rows of a
// head with such a row redo, as when each head had a block of its own; the others take part in the fetches and barriers.
// One row of a call out of range (K 65536, 16 on 2 heads, Q 128, D 64: blocks of 512 rows laid end to end):
// 156 us, with none 105, with every wave of the block redoing 198, head by head 174.  Writes (m, log2 l) per row, or
// (m, l) per (split, row) when the keys are split; the column pass merges the splits.
// PRE: see the column pass.  The common sweep runs its stages below a.pre_end on Q * c rounded to fp16 (then the
// rest on the raw operand) and accepts row sums below 2^20 only; a block that leaves the range reloads the raw
// operand for its stabilised sweeps, all waves of it: the column pass then takes the raw operand for the whole unit.
template <int D, int NB, int WAVES, bool BF, bool PRE, bool FOLD>
__global__ __launch_bounds__(64 * WAVES, 2) void fcs_rowstream_kernel(const Args a)
{
    static_assert(!PRE || (!BF && D == 64), "the pre-scaled variant exists for fp16 operands and 64-wide heads");
    constexpr int THREADS = 64 * WAVES;
    constexpr int NT = D / 16;
    constexpr int NTA = NT < 8 ? NT : 8;
    constexpr int KT = kStageKeys;
    constexpr int NA = KT / 32;
    constexpr int ROWS_W = 32 * NB;
    constexpr int BLOCK_ROWS = WAVES * ROWS_W;
    constexpr int ROW_BYTES = D * 2;
    constexpr int PPR = D / 8;
    constexpr int STAGE_BYTES = KT * ROW_BYTES;
    constexpr int IPW = KT * PPR / THREADS;
    constexpr int NS = row_ring_slots(D, WAVES);
    constexpr int RP = 33;  // floats per row of the transpose buffer
    static_assert(IPW >= 1 && KT * PPR == IPW * THREADS, "a stage is a whole number of DMA instructions per wave");
    static_assert(NS >= 3 && NS <= 4, "ring depth");
    __shared__ __attribute__((aligned(16))) char ring[NS * STAGE_BYTES];
    __shared__ __attribute__((aligned(16))) float red[WAVES * 32 * RP];  // wave-private [32 rows][RP]
    __shared__ __attribute__((aligned(16))) float mrow[BLOCK_ROWS];      // row maxima of the stabilised sweeps
    __shared__ int bad_s[WAVES];
    __shared__ int2 redo_s[kRedoHeads<PRE, FOLD> ? WAVES : 1];  // of such a wave: the rows that are redone, from .x to one before .y

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int bx, chunk, bh;  // row blocks of one (key split, head) read the same keys: same XCD
    xcd_contiguous_block((int)blockIdx.x, a.n_qblk, a.n_chunks, a.B * a.v_heads, bx, chunk, bh);  // a one-dimensional grid: no axis limit
    const int b = bh / a.v_heads, h = bh - b * a.v_heads;
    const int row0 = bx * BLOCK_ROWS, qw0 = row0 + wave * ROWS_W;
    const float cmul = a.c;

    // key range of this block: its split, cut at the last key any of its rows may see
    const int kc0 = chunk * a.chunk_keys;
    int kc1 = min(a.Sk, kc0 + a.chunk_keys);
    if (a.causal) kc1 = min(kc1, a.k_past + rows_past<FOLD>(a, row0 + BLOCK_ROWS));
    const int nst = (kc1 > kc0) ? (kc1 - kc0 + KT - 1) / KT : 0;

    uint32_t g_off[IPW];
#pragma unroll
    for (int j = 0; j < IPW; ++j) {
        const int P = (wave * IPW + j) * 64 + lane;
        const int row = P / PPR, pos = P % PPR;
        g_off[j] = (uint32_t)row * (uint32_t)(a.ks_s * 2) + (uint32_t)((pos ^ row_swizzle<D>(row)) * 16);
    }
    char *ring_w = ring + wave * (IPW * 1024);
    uint32_t take[NTA];
#pragma unroll
    for (int t = 0; t < NTA; ++t)
        take[t] = lds_addr(ring) + (uint32_t)(n * ROW_BYTES + (((2 * t + g) ^ row_swizzle<D>(n)) * 16));

    half8 qf[NB][NT];
    auto load_q = [&](bool scaled) {  // this wave's query rows: pre-scaled, or raw with the scale's sign
        int lane_o = lane;
        asm volatile("" : "+v"(lane_o));  // addresses are formed here, not kept for a second call
        const int n_o = lane_o & 31, g_o = lane_o >> 5;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const _Float16 *row = q_row_ptr<FOLD>(a, b, h, qw0 + nb * 32 + n_o) + g_o * 8;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                half8 v = kZero8;
                if (t * 16 + g_o * 8 < a.D) v = load8(row + t * 16);
                if (PRE && scaled) qf[nb][t] = prescale(v, a.negate ? -a.c : a.c);
                else qf[nb][t] = a.negate ? flip_sign(v) : v;
            }
        }
    };
    // leading stages of the block that run on the pre-scaled operand in the common sweep (block-uniform)
    const int n_pre = PRE ? min(nst, max(0, (a.pre_end - kc0) / KT)) : 0;
    load_q(n_pre > 0);
    const char *kp = reinterpret_cast<const char *>(a.k + (int64_t)b * a.ks_b +
                                                    (int64_t)kv_head(h, a.kv_group, a.kv_magic) * a.ks_h);
    const int64_t k_row_b = a.ks_s * 2;
    const int kp_eff = a.causal ? a.k_past : 0x3fffffff - a.Sq;
    const int thr_wave_min = a.causal ? min(a.k_past + rows_first<FOLD>(a, qw0, ROWS_W), a.Sk - 1) : a.Sk - 1;
    const int thr_wave_max = a.causal ? a.k_past + (FOLD ? a.q_rows : qw0 + ROWS_W) - 1 : a.Sk - 1;
    const int n_plain = plain_stages(kc0, nst, thr_wave_min), n_seen = seen_stages(kc0, nst, thr_wave_max);

    auto fetch_stage = [&](int st, int slot) {
        const int kb = kc0 + min(st, nst - 1) * KT;
        char *dst = ring_w + slot * STAGE_BYTES;
        if (__builtin_expect(kb + KT <= a.Sk && a.D == D, 1)) {
            const char *src = kp + (int64_t)kb * k_row_b;
#pragma unroll
            for (int j = 0; j < IPW; ++j) dma16(src + g_off[j], dst + j * 1024);
        } else {
            int lane_o = lane;
            asm volatile("" : "+v"(lane_o));
#pragma unroll
            for (int j = 0; j < IPW; ++j) {
                const int P = (wave * IPW + j) * 64 + lane_o;
                const int row = P / PPR, pos = P % PPR;
                const int piece = pos ^ row_swizzle<D>(row);
                const char *src = kp + (int64_t)min(kb + row, a.Sk - 1) * k_row_b + piece * 16;
                if (piece * 8 >= a.D) src = reinterpret_cast<const char *>(g_zero_piece);
                dma16(src, dst + j * 1024);
            }
        }
    };
    half8 kf[NT];
    auto take_frag = [&](auto off_c, half8 (&dst)[NT]) {
        constexpr int OFF = decltype(off_c)::value;
        constexpr int IMM = (OFF < 65536 - 256) ? OFF : 0;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const uint32_t ad = take[t % NTA] + (uint32_t)(OFF - IMM);
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst[t]) : "v"(ad), "n"(IMM + t / NTA * 256) : "memory");
        }
    };
    auto take_frag_at = [&](int off, half8 (&dst)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const uint32_t ad = take[t % NTA] + (uint32_t)off;
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst[t]) : "v"(ad), "n"(t / NTA * 256) : "memory");
        }
    };
    auto frag_wait = [&](half8 (&dst)[NT]) {
#pragma unroll
        for (int t0 = 0; t0 < NT; t0 += 4)
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(dst[t0]), "+v"(dst[t0 + 1]), "+v"(dst[t0 + 2]), "+v"(dst[t0 + 3])::"memory");
    };

    float rs[NB][16];      // running per-row value (sum or maximum) over this lane's keys
    float nmax[NB][16];    // -m_i of the rows in accumulator layout (stabilised sum sweep only)

    // One sweep over the stages [s0, s1) of the block's keys.  MAXOP: rs = max of the visible scores; else
    // rs += 2^(score * c) over the visible keys.  SHIFT: the row's -m_i (in `nmax`) is added to the score before
    // the scale.  SCALED: the operand in `qf` is the pre-scaled one.  The accumulators always start at 0, so that
    // every sweep, and the column pass for these rows, sees the very same score bits.
    auto reset_rows = [&](auto max_c) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) rs[nb][i] = decltype(max_c)::value ? kNegBig : 0.f;
    };
    // A wave that is not `active` takes part in the fetches and barriers alone.
    auto sweep = [&](auto max_c, auto shift_c, auto scaled_c, const int s0, const int s1, const bool active) {
        constexpr bool MAXOP = decltype(max_c)::value;
        constexpr bool SHIFT = decltype(shift_c)::value;
        constexpr bool SCALED = decltype(scaled_c)::value;
        static_assert(!SCALED || (PRE && !MAXOP && !SHIFT), "only the common sweep of the pre-scaled variant");
        constexpr int TILES = NA * NB;
        static_assert(NA == 2 && TILES % 2 == 0, "fragment offsets and the two alternating accumulators");
        if (s1 <= s0) return;  // block-uniform
#pragma unroll
        for (int st = 0; st < NS - 1; ++st) fetch_stage(s0 + st, st);
        FCS_WAIT_VM((NS - 3) * IPW);
        block_sync();
        auto drain_plain = [&](const floatx16 &sc, int nb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if (MAXOP) rs[nb][i] = fmaxf(rs[nb][i], sc[i]);
                else rs[nb][i] += SCALED ? fast_exp2(sc[i]) : fast_exp2((SHIFT ? sc[i] + nmax[nb][i] : sc[i]) * cmul);
            }
        };
        auto drain_masked = [&](const floatx16 &sc, int kb_t, int na, int nb) {
            const int key = kb_t + na * 32 + n;
            int rel = (key < a.Sk) ? key - kp_eff - (qw0 + 4 * g) : 0x3fffffff;
            asm volatile("" : "+v"(rel));
            mask_rows<FOLD>(a, qw0 + nb * 32, 4 * g, rel, [&](auto ahead) {
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const bool vis = rel + ahead(i) <= nb * 32 + 8 * (i >> 2) + (i & 3);
                    if (MAXOP) rs[nb][i] = fmaxf(rs[nb][i], vis ? sc[i] : kNegBig);
                    else rs[nb][i] += vis ? (SCALED ? fast_exp2(sc[i]) : fast_exp2((SHIFT ? sc[i] + nmax[nb][i] : sc[i]) * cmul)) : 0.f;
                }
            });
        };
        const floatx16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        auto chain = [&](int nb) {
            floatx16 c = mfma16<BF>(qf[nb][0], kf[0], zero16);
#pragma unroll
            for (int t = 1; t < NT; ++t) c = mfma16<BF>(qf[nb][t], kf[t], c);
            return c;
        };

        // ---- the plain stream (see the column pass): stages [s0, sp)
        const int sp = active ? min(s1, max(s0, n_plain)) : s0;
        if (sp > s0) {
            take_frag(std::integral_constant<int, 0>{}, kf);
            floatx16 acc[2];
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[0][i] = acc[1][i] = 0.f;
            auto stage = [&](int st, auto slot_c) {
                constexpr int SLOT = decltype(slot_c)::value;
                const bool first = SLOT == 0 && st == s0;
                if (!first) {
                    FCS_WAIT_VM((NS - 3) * IPW);
                    block_barrier();
                }
                fetch_stage(st + NS - 1, (SLOT + NS - 1) % NS);
#pragma unroll
                for (int q = 0; q < TILES; ++q) {
                    const int na = q / NB, nb = q % NB;
                    if (nb == 0) frag_wait(kf);
                    acc[q & 1] = chain(nb);
                    asm volatile("" : "+v"(acc[0]), "+v"(acc[1]));
                    if (nb == NB - 1) {
                        if (na == 0) take_frag(std::integral_constant<int, SLOT * STAGE_BYTES + 32 * ROW_BYTES>{}, kf);
                        else take_frag(std::integral_constant<int, ((SLOT + 1) % NS) * STAGE_BYTES>{}, kf);
                    }
                    if (q > 0 || !first) drain_plain(acc[(q + 1) & 1], (q > 0) ? (q - 1) % NB : NB - 1);
                }
            };
            for (int st0 = s0; st0 < sp; st0 += NS) {
                stage(st0, std::integral_constant<int, 0>{});
                if (st0 + 1 < sp) stage(st0 + 1, std::integral_constant<int, 1>{});
                if (st0 + 2 < sp) stage(st0 + 2, std::integral_constant<int, 2>{});
                if (NS > 3 && st0 + 3 < sp) stage(st0 + 3, std::integral_constant<int, 3 % NS>{});
            }
            frag_wait(kf);
            drain_plain(acc[(TILES - 1) & 1], NB - 1);
        }

        // ---- the rest, as in the column pass
        const int sv = active ? min(s1, max(sp, n_seen)) : s0;
        int slot = (sp - s0) % NS;
        auto enter_stage = [&](int st) {
            if (st > s0) {
                FCS_WAIT_VM((NS - 3) * IPW);
                block_barrier();
            }
            fetch_stage(st + NS - 1, (slot == 0) ? NS - 1 : slot - 1);
            slot = (slot + 1 == NS) ? 0 : slot + 1;
        };
        if constexpr (NB == 1 && D <= 128) {
            if (sv > sp) {
                floatx16 acc[2];
                acc[0] = acc[1] = zero16;
                if (sp == s0) take_frag(std::integral_constant<int, 0>{}, kf);
                frag_wait(kf);
#pragma unroll 1
                for (int st = sp; st < sv; ++st) {
                    const int kb = kc0 + st * KT, here = slot * STAGE_BYTES;
                    enter_stage(st);
                    frag_wait(kf);
                    acc[0] = chain(0);
                    asm volatile("" : "+v"(acc[0]), "+v"(acc[1]));
                    take_frag_at(here + 32 * ROW_BYTES, kf);
                    frag_wait(kf);
                    acc[1] = chain(0);
                    asm volatile("" : "+v"(acc[0]), "+v"(acc[1]));
                    take_frag_at(slot * STAGE_BYTES, kf);
                    drain_masked(acc[0], kb, 0, 0);
                    drain_masked(acc[1], kb, 1, 0);
                }
                frag_wait(kf);
            }
        } else {
            for (int st = sp; st < sv; ++st) {
                const int kb = kc0 + st * KT, here = slot * STAGE_BYTES;
                enter_stage(st);
#pragma unroll 1
                for (int s = 0; s < TILES / 2; ++s) {
                    floatx16 acc[2];
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        if (NB == 1 || q == 0) {
                            take_frag_at(here + (NB == 1 ? q : s) * 32 * ROW_BYTES, kf);
                            frag_wait(kf);
                        }
                        acc[q] = chain(NB == 1 ? 0 : q);
                    }
#pragma unroll
                    for (int q = 0; q < 2; ++q) drain_masked(acc[q], kb, NB == 1 ? q : s, NB == 1 ? 0 : q);
                }
            }
        }
        for (int st = sv; st < s1; ++st) enter_stage(st);
        FCS_WAIT_VM(0);
        block_sync();  // the ring may be refilled by the next sweep
    };

    // rs[nb][*] over the 32 key lanes: every lane gets the value of row nb * 32 + (lane % 32) of this wave.
    // Fixed order of additions.  (No DMA is in flight here, so these are ordinary LDS accesses.)
    float *red_w = red + wave * (32 * RP);
    auto fold_lanes = [&](auto max_c, float (&tot)[NB]) {
        constexpr bool MAXOP = decltype(max_c)::value;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) red_w[(8 * (i >> 2) + 4 * g + (i & 3)) * RP + n] = rs[nb][i];
            __builtin_amdgcn_wave_barrier();
            float v = MAXOP ? kNegBig : 0.f;  // each half-wave takes 16 of the row's 32 lanes' values
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                const float x = red_w[n * RP + g * 16 + j];
                v = MAXOP ? fmaxf(v, x) : v + x;
            }
            const float o = __shfl_xor(v, 32);
            tot[nb] = MAXOP ? fmaxf(v, o) : (g == 0 ? v + o : o + v);  // lower half first in both halves
            __builtin_amdgcn_wave_barrier();
        }
    };

    // ---- common path: no max subtraction; the pre-scaled stages first, then the raw ones
    reset_rows(std::false_type{});
    if constexpr (PRE) {
        sweep(std::false_type{}, std::false_type{}, std::true_type{}, 0, n_pre, true);
        if (n_pre > 0 && n_pre < nst) load_q(false);
    }
    sweep(std::false_type{}, std::false_type{}, std::false_type{}, n_pre, nst, true);
    float lt[NB], m_row[NB];
    fold_lanes(std::false_type{}, lt);
    bool has[NB], out[NB], bad = false;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int qi = rows_first<FOLD>(a, qw0 + nb * 32 + n, 1);
        const int thr = a.causal ? min(a.k_past + qi, a.Sk - 1) : a.Sk - 1;  // last key this row sees
        has[nb] = (nst > 0) && (kc0 <= thr);
        // ceiling 2^110 rather than 2^120: up to 512 key splits of a row are added up by the column pass
        out[nb] = has[nb] && !(lt[nb] >= 8.2718061e-25f && lt[nb] < (n_pre > 0 ? kRowSumHiPre : 1.2980742e+33f));
        bad = bad || out[nb];
        m_row[nb] = has[nb] ? 0.f : kNegBig;  // an empty split must not set the merged maximum
        if (!has[nb]) lt[nb] = 0.f;
    }
    {
        const bool wbad = __builtin_amdgcn_ballot_w64(bad) != 0;
        if (lane == 0) bad_s[wave] = wbad ? 1 : 0;
        if constexpr (kRedoHeads<PRE, FOLD>) {
            if (wbad) {  // rows of the heads from the wave's first such row to its last
                uint64_t set = 0;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)  // both half-waves hold the same rows
                    set |= (uint64_t)(uint32_t)__builtin_amdgcn_ballot_w64(out[nb]) << (32 * nb);
                const int first = fold_head(qw0 + __builtin_ctzll(set), a.fold_magic) * a.q_rows;
                const int past = (fold_head(qw0 + 63 - __builtin_clzll(set), a.fold_magic) + 1) * a.q_rows;
                if (lane == 0) redo_s[wave] = int2{first, past};
            }
        }
        block_sync();
        int any = 0;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) any |= bad_s[w];
        bad = any != 0;  // block-uniform
    }

    // ---- rare: row maxima first, then sums with the maximum subtracted before the scale
    if (bad) {
        bool redo = true;  // wave-uniform
        if constexpr (kRedoHeads<PRE, FOLD>) {
            redo = false;
            for (int w = 0; w < WAVES; ++w)
                if (bad_s[w]) redo = redo || (redo_s[w].x < qw0 + ROWS_W && redo_s[w].y > qw0);
            redo = __builtin_amdgcn_readfirstlane(redo) != 0;
        }
        if (PRE) load_q(false);
        reset_rows(std::true_type{});
        sweep(std::true_type{}, std::false_type{}, std::false_type{}, 0, nst, redo);
        float mx[NB];
        fold_lanes(std::true_type{}, mx);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (!has[nb]) mx[nb] = 0.f;  // no visible key in this split: every exponential is masked anyway
            if (g == 0) mrow[wave * ROWS_W + nb * 32 + n] = mx[nb];
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int i = 0; i < 16; ++i) nmax[nb][i] = -mrow[wave * ROWS_W + nb * 32 + 8 * (i >> 2) + 4 * g + (i & 3)];
        reset_rows(std::false_type{});
        sweep(std::false_type{}, std::true_type{}, std::false_type{}, 0, nst, redo);
        float ls[NB];
        fold_lanes(std::false_type{}, ls);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (!redo) continue;  // m = 0 and the sum of the common path stand
            m_row[nb] = has[nb] ? mx[nb] : kNegBig;
            lt[nb] = has[nb] ? ls[nb] : 0.f;
        }
    }

    // ---- store: the lower half-wave holds one row per lane
    if (g == 0) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int qi = qw0 + nb * 32 + n;  // < rows_pad by construction
            float2 v;
            v.x = m_row[nb];
            if (a.n_chunks == 1) {
                v.y = fast_log2(lt[nb]);
                a.lse[(int64_t)bh * a.rows_pad + qi] = v;
            } else {
                v.y = lt[nb];
                a.ml[((int64_t)bh * a.n_chunks + chunk) * a.rows_pad + qi] = v;
            }
        }
    }
}

// ------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------
// Both passes must agree on the pre-scaled variant: fp16 operands, 64-wide kernels, |scale| <= 1/8, and
// at least 16384 (head, row) pairs averaged into every output that is computed from pre-scaled scores (the
// rounding of Q * c to fp16 perturbs every score by about 2^-12 relative; over that many rows its effect on a
// mean stays below 2e-4 relative at unit-variance inputs).  Of a causal call only the keys that every row sees
// qualify, in whole 64-key stages (Args::pre_end): its last keys are seen by a handful of rows only, and there the
// perturbation shows undiminished (measured 1e-3 relative at four times unit-variance inputs).
// (128-wide heads gain nothing from it: there the matrix pipe has twice the work per score and the kernels are no
// longer bound by the exponent's VALU work alone: B 1, H 16, S 8192, D 128 548 against 552 us, the causal
// H 32, Q 512, K 65536, D 128 622 against 610 us.)
inline bool stream_prescaled(const Plan &p, const Args &a)
{
    return !p.bf16 && p.Dp == 64 && a.c != 0.f && fabsf(a.c) <= 0.1251f * 1.44269504f && (long)p.H * p.q_rows >= 16384 &&
           a.pre_end >= 4 * kStageKeys;
}

template <int D, int NB, int WAVES, bool BF, bool FOLD>
static hipError_t launch_cfg(const Plan &p, const Args &a, hipStream_t st)
{
    const dim3 grid((unsigned)((long)p.c_nchunks * p.c_groups * p.B));
    if constexpr (D == 64 && !BF) {
        if (stream_prescaled(p, a)) {
            hipLaunchKernelGGL((fcs_colstream_kernel<D, NB, WAVES, BF, true, FOLD>), grid, dim3(64 * WAVES), 0, st, a);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((fcs_colstream_kernel<D, NB, WAVES, BF, false, FOLD>), grid, dim3(64 * WAVES), 0, st, a);
    return hipGetLastError();
}

template <int D, bool BF, bool FOLD>
static hipError_t launch_colstream_d(const Plan &p, const Args &a, hipStream_t st)
{
    if constexpr (D <= 128) {
        if (p.c_nb == 2 && p.c_waves == 8) return launch_cfg<D, 2, 8, BF, FOLD>(p, a, st);
        if (p.c_nb == 2 && p.c_waves == 4) return launch_cfg<D, 2, 4, BF, FOLD>(p, a, st);
        if (p.c_nb == 1 && p.c_waves == 4) return launch_cfg<D, 1, 4, BF, FOLD>(p, a, st);
    } else {
        if (p.c_nb == 1 && p.c_waves == 8) return launch_cfg<D, 1, 8, BF, FOLD>(p, a, st);
        if (p.c_nb == 1 && p.c_waves == 4) return launch_cfg<D, 1, 4, BF, FOLD>(p, a, st);
    }
    return hipErrorInvalidValue;
}

template <int D, int NB, int WAVES, bool BF, bool FOLD>
static hipError_t launch_rows_cfg(const Plan &p, const Args &a, hipStream_t st)
{
    const dim3 grid((unsigned)((long)p.n_qblk * p.n_chunks * p.B * p.v_heads));
    if constexpr (D == 64 && !BF) {
        if (stream_prescaled(p, a)) {
            hipLaunchKernelGGL((fcs_rowstream_kernel<D, NB, WAVES, BF, true, FOLD>), grid, dim3(64 * WAVES), 0, st, a);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((fcs_rowstream_kernel<D, NB, WAVES, BF, false, FOLD>), grid, dim3(64 * WAVES), 0, st, a);
    return hipGetLastError();
}

template <int D, bool BF, bool FOLD>
static hipError_t launch_rowstream_d(const Plan &p, const Args &a, hipStream_t st)
{
    if constexpr (D <= 128) {
        if (p.qw == 64 && p.k1_waves == 8) return launch_rows_cfg<D, 2, 8, BF, FOLD>(p, a, st);
        if (p.qw == 64 && p.k1_waves == 4) return launch_rows_cfg<D, 2, 4, BF, FOLD>(p, a, st);
    }
    if (p.qw == 32 && p.k1_waves == 4) return launch_rows_cfg<D, 1, 4, BF, FOLD>(p, a, st);
    return hipErrorInvalidValue;
}

template <bool FOLD>
hipError_t launch_rowstream_f(const Plan &p, const Args &a, hipStream_t st)
{
    if (p.bf16)
        return (p.Dp == 64) ? launch_rowstream_d<64, true, FOLD>(p, a, st)
                            : (p.Dp == 128) ? launch_rowstream_d<128, true, FOLD>(p, a, st) : launch_rowstream_d<256, true, FOLD>(p, a, st);
    return (p.Dp == 64) ? launch_rowstream_d<64, false, FOLD>(p, a, st)
                        : (p.Dp == 128) ? launch_rowstream_d<128, false, FOLD>(p, a, st) : launch_rowstream_d<256, false, FOLD>(p, a, st);
}

template <bool FOLD>
hipError_t launch_colstream_f(const Plan &p, const Args &a, hipStream_t st)
{
    if (p.bf16)
        return (p.Dp == 64) ? launch_colstream_d<64, true, FOLD>(p, a, st)
                            : (p.Dp == 128) ? launch_colstream_d<128, true, FOLD>(p, a, st) : launch_colstream_d<256, true, FOLD>(p, a, st);
    return (p.Dp == 64) ? launch_colstream_d<64, false, FOLD>(p, a, st)
                        : (p.Dp == 128) ? launch_colstream_d<128, false, FOLD>(p, a, st) : launch_colstream_d<256, false, FOLD>(p, a, st);
}

}  // namespace fcs
