// Attention column means on gfx950 (MI355X): the kernels of the general two-pass path.  The column pass comes first.
// (Causal calls of one batch entry and up to 2048 keys are mostly served by fcs_tall.hip; where such a size is quoted below, it was
// measured here.)
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
// The keys are cut into chunks (at most col_chunk_max(), the LDS accumulator).  The work is a line of stages: batch
// entry, chunk, head, row block, stage; every workgroup takes an equal share of it (StageLine in fcs_plan.h), walks over the
// (head, row block) units of its share, re-streaming the chunk for each, and leaves one partial slab per chunk that it
// touched: the waves' slices added in wave order.  What bounds a call that is cut unit by unit is its longest
// workgroup: of a causal prompt the row blocks see 8, 16, .. 64 stages, and of 144 or 304 equal units every second or the
// last compute units have nothing to do.  Both passes on the line, against whole units (this pass and pass 1, us per
// call): causal H 32, S 4096, D 128 bf16 229 -> 163; H 12, S 5242, D 64 178 -> 124; H 12, S 4491, D 64 bf16 146 -> 102;
// H 16, S 9459, D 64 571 -> 467; H 8, S 4435, D 128 bf16 causal 97 -> 69.  Where whole units of one length fill
// the chip evenly the plan keeps to them, one to a workgroup (ONE: the walk and its state are compiled out; a small call spends
// half its time before the first stage, and cold instructions are a good part of that).  us per call, the same shares with the
// walk -> without: causal H 32, Q 128, K 4096, D 128 29.1 -> 22.9, K 16384 60.1 -> 57.6; H 32, S 634 30.8 -> 25.7; H 8, Q 512,
// K 4096, D 256 35.1 -> 31.0; H 16, S 4096, D 64 90.9 -> 86.7; 32 on 8 heads laid end to end, Q 64, K 8192 53.3 -> 53.1.
// At a unit's start the first stages, the row statistics and the query rows are requested together, and nothing is
// requested past a unit's last stage.  Causal alignment  j <= k_past + i  (reference:
// flash_colsum/kernel_causal.py:39,57,113): the stage loop stops at the last key any row of the
// unit sees, only stages on the diagonal (or past the last key) take the masked code path.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fcs_device.h"
#include "fcs_kernels.h"
#include "fcs_rowfold.h"

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
constexpr uint32_t kPastDim = 0xffffffffu;  // in the place of such a piece's offset

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

// Which 16-byte piece of its row a lane of half-wave g takes for MFMA step t (the contraction may run in any order, as long as
// both operands take the same one): four steps take 64 consecutive bytes of a row.
template <int NTA>
__host__ __device__ constexpr int piece_of(int t, int g)
{
    return t % NTA + NTA * g + 2 * NTA * (t / NTA);
}

// The stationary rows.  A lane needs pieces of its own row, but four neighbouring lanes first read 64 consecutive bytes of one
// of their four rows after the other: an access of four lanes to four rows takes the address path four times as long (a block of
// 512 rows of 128 channels had its rows 5 .. 9 us after its start, the first stages long before).  Row pass with 32 bytes of a
// row per access, then with this, against the same kernel on the same box: H 32, Q 512, K 65536, D 128 0.985 and 0.977 of its
// time, H 16, S 8192, D 64 0.978 and 0.967.  load_quads leaves row
// (lane & ~3) + j in f[nb][4 * i + j], pieces 4 * i ..; quad_transpose then hands every lane its own row.
template <int D, int NB, bool FOLD>
__device__ __forceinline__ void load_quads(const Args &a, int b, int h, int first_row, int lane, half8 (&f)[NB][D / 16])
{
    constexpr int NT = D / 16, NTA = NT < 8 ? NT : 8;
    const int n4 = lane & 28, q = lane & 3, g = lane >> 5;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const _Float16 *row = q_row_ptr<FOLD>(a, b, h, first_row + nb * 32 + n4 + j);
#pragma unroll
            for (int i = 0; i < NT / 4; ++i) {
                // (narrower heads: the row's last piece again in the place of those past it, see zero_past_dim)
                const int at = (piece_of<NTA>(4 * i, g) + q) * 8;
                f[nb][4 * i + j] = load8(row + min(at, a.D - 8));
            }
        }
}
// 4 x 4 transposes within four neighbouring lanes: two rounds of exchanges, with the lane 1 away and with the lane 2 away.
// v_cndmask_b32 with the quad permutation on its first source does select and exchange in one; a register that a vector
// instruction wrote may be read through a permutation two wait states later.
#define FCS_QUAD_PICK(DST, OTHER, OWN, PERM) "v_cndmask_b32_dpp " DST ", " OTHER ", " OWN ", vcc quad_perm:" PERM " row_mask:0xf bank_mask:0xf\n\t"
template <int NT>
__device__ __forceinline__ void quad_transpose(half8 (&f)[NT])
{
    const uint64_t even = 0x5555555555555555ull, low = 0x3333333333333333ull;
#pragma unroll
    for (int i = 0; i < NT; i += 4) {
        uint4v x[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) x[j] = __builtin_bit_cast(uint4v, f[i + j]);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            uint32_t p0 = x[0][c], p1 = x[1][c], p2 = x[2][c], p3 = x[3][c], y0, y1, y2, y3;
            asm("s_mov_b64 vcc, %8\n\ts_nop 1\n\t"                            // even lanes keep rows 0 and 2
                FCS_QUAD_PICK("%4", "%1", "%0", "[1,0,3,2]") FCS_QUAD_PICK("%6", "%3", "%2", "[1,0,3,2]")
                "s_not_b64 vcc, vcc\n\t"                                        // odd lanes rows 1 and 3
                FCS_QUAD_PICK("%5", "%0", "%1", "[1,0,3,2]") FCS_QUAD_PICK("%7", "%2", "%3", "[1,0,3,2]")
                "s_mov_b64 vcc, %9\n\ts_nop 1\n\t"                            // then the same two lanes apart
                FCS_QUAD_PICK("%0", "%6", "%4", "[2,3,0,1]") FCS_QUAD_PICK("%1", "%7", "%5", "[2,3,0,1]")
                "s_not_b64 vcc, vcc\n\t"
                FCS_QUAD_PICK("%2", "%4", "%6", "[2,3,0,1]") FCS_QUAD_PICK("%3", "%5", "%7", "[2,3,0,1]")
                : "+v"(p0), "+v"(p1), "+v"(p2), "+v"(p3), "=&v"(y0), "=&v"(y1), "=&v"(y2), "=&v"(y3)
                : "s"(even), "s"(low)
                : "vcc", "scc");
            x[0][c] = p0;
            x[1][c] = p1;
            x[2][c] = p2;
            x[3][c] = p3;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) f[i + j] = __builtin_bit_cast(half8, x[j]);
    }
}
#undef FCS_QUAD_PICK
// channels past the tensor's head dim are zeros
template <int NT>
__device__ __forceinline__ void zero_past_dim(half8 (&f)[NT], int dim, int g)
{
    constexpr int NTA = NT < 8 ? NT : 8;
#pragma unroll
    for (int t = 0; t < NT; ++t)
        if (piece_of<NTA>(t, g) * 8 >= dim) f[t] = kZero8;
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

// A stage with n - 1 more behind it in its stream is entered (n > 0): the one behind it has landed once at most the stages
// requested after that are outstanding, NS - 3 of them, or none at the stream's end.  (Other loads in flight make it wait longer.)
template <int NS, int IPW>
__device__ __forceinline__ void wait_stages(int n)
{
    if (NS > 3 && n >= NS - 1) FCS_WAIT_VM((NS - 3) * IPW);
    else FCS_WAIT_VM(0);
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
// Column pass: log2 of a row's sum in score units, log2(l) / c, overflows below a scale of 1e-37; from here on down the form without
// it is taken (bf16 scores reach 2^127, so that such a scale still tells keys apart).
constexpr float kTinyScale = 1e-30f;

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
// ONE: a workgroup has one chunk of one unit (see the plan).
template <int D, int NB, int WAVES, bool BF, bool PRE, bool FOLD, bool ONE>
__global__ __launch_bounds__(64 * WAVES, 2) void fcs_colstream_kernel(const Args a)
{
    // A workgroup with one chunk of one unit streams the stages that all its rows see backwards: pass 1 has just read the same keys forwards, and
    // its last ones are what the Infinity Cache surely still holds.  (The L2s hold nothing from kernel to kernel: their fetch traffic is all of the
    // keys either way.)  us per call on changing keys, forwards -> backwards, D 128: H 32 Q 128 K 16384 69.5 -> 68.0 (bf16 61.7 -> 60.6), K 8192 35.3 -> 34.1,
    // K 32768 114.3 -> 113.8, 4 x 32 heads on 8, Q 64 K 8192 51.7 -> 49.6 (it varies by 2 % from box to box); same bits (a key's sums do not depend on the
    // stages' order).  Alternating directions over the units of a walk gained nothing (S 4096 167.9 and 167.8, S 8192 D 64 bf16 353 and 357).
    constexpr bool REV = ONE && !PRE;
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
    constexpr int ROWS1 = D == 256 ? 128 : BLOCK_ROWS;  // pass 1's row blocks
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
    fetch_args(a);
    int share = xcd_contiguous((int)blockIdx.x, a.c_blocks);  // neighbours on the line run on one XCD
    const float cmul = (a.c == 0.f) ? 1.f : a.c;       // scale 0: Q is zeroed instead and n_i = -log2 l_i

    const float inv_c = __builtin_amdgcn_rcpf(cmul);
    const bool tiny = cmul < kTinyScale;
    float *colw_w = colw + wave * CHUNK;  // this wave's slice of the column accumulator

    // ---- DMA geometry: piece P of a stage goes to LDS byte 16 * P; it is piece pos ^ swizzle(row)
    // of stage row `row`, so that row r keeps piece p at position p ^ swizzle(r)
    uint32_t g_off[IPW];   // byte offset of this lane's piece from the stage's first key row (dense stage)
#pragma unroll
    for (int j = 0; j < IPW; ++j) {
        const int P = (wave * IPW + j) * 64 + lane;
        const int row = P / PPR, pos = P % PPR;
        const int piece = pos ^ row_swizzle<D>(row);
        g_off[j] = (D == 128 || piece * 8 < a.D) ? (uint32_t)row * (uint32_t)(a.ks_s * 2) + (uint32_t)(piece * 16) : kPastDim;
    }
    char *ring_w = ring + wave * (IPW * 1024);  // where this wave's pieces of a stage land inside a slot
    // operand read-back: lane (n, g) takes, for MFMA step t, piece piece_of(t, g) of row n (+ 32 per key fragment)
    uint32_t take[NTA];
#pragma unroll
    for (int t = 0; t < NTA; ++t)
        take[t] = lds_addr(ring) + (uint32_t)(n * ROW_BYTES + ((piece_of<NTA>(t, g) ^ row_swizzle<D>(n)) * 16));

    // ---- where this workgroup's share of the line starts: batch entry, chunk, head, row block, place in it
    int b, cx, h = 0, rb = 0, at = 0, left = 0x7fffffff;  // left: places of the share that are still to do
    if constexpr (ONE) {
        // The chunks of a unit side by side: of causal units the last ones are empty, and every XCD gets its part of them
        // (H 32, Q = K 634, D 128: 15.6 us with a chunk's units side by side).
        b = a.by_heads.quot(a.c_by_blocks.quot(a.c_by_chunks.quot(share, cx), rb), h);
        share = ((b * (int)a.c_by_chunks.d + cx) * a.v_heads + h) * a.c_nrb + rb;
    } else if (a.c_direct) {
        b = a.c_by_chunks.quot(share, cx);
    } else if (a.c_unit > 1) {  // counted in chunks of units
        const int pos = share * a.c_seg;
        left = min(a.c_seg, a.c_len - pos);
        b = a.c_by_chunks.quot(a.by_heads.quot(a.c_by_blocks.quot(pos, rb), h), cx);
    } else {
        int pos = share * a.c_seg;
        left = min(a.c_seg, a.c_len - pos);
        b = a.c_by_batch.quot(pos, pos);
        // The chunk: those that every row block sees to its end are alike, from there on one after the other.  (Adding up all
        // chunks before each of them was 20 % of H 8, Q 1024, K 262144, D 128, 1549 us against 1291 head by head in whole units.)
        cx = min(a.c_by_chunks.quot(pos), a.c_every - (a.c_every * a.c_cs > a.c_line.n(0) ? 1 : 0));
        int pairs = cx * a.c_nrb, lo = a.c_line.sum(a.c_nrb, cx * a.c_cs) + pairs * a.c_line.start, hi;
        for (;; ++cx, lo = hi) {
            pairs += a.c_line.sees(a.c_nrb, a.c_cs, cx);
            hi = a.c_line.sum(a.c_nrb, (cx + 1) * a.c_cs) + pairs * a.c_line.start;
            if (pos < a.v_heads * hi) break;
        }
        pos -= a.v_heads * lo;
        const int per_h = hi - lo;
        h = (int)((float)pos * __builtin_amdgcn_rcpf((float)per_h));  // the head or a neighbour of it
        h = __builtin_amdgcn_readfirstlane(h);
        for (pos -= h * per_h; pos < 0; --h) pos += per_h;
        for (; pos >= per_h; ++h) pos -= per_h;
        for (;; ++rb) {
            const int n_rb = a.c_line.between(rb, cx * a.c_cs, (cx + 1) * a.c_cs), len = n_rb > 0 ? n_rb + a.c_line.start : 0;
            if (pos < len) break;
            pos -= len;
        }
        at = pos;
    }

    for (;;) {  // the chunks that the share touches
    const int ck0 = cx * a.c_chunk;                    // first key of the chunk
    const int c1 = min(a.Sk, ck0 + a.c_chunk);         // one past its last key
    bool cleared = false;
    auto clear_slice = [&]() {
        const floatx4 zero4 = {0.f, 0.f, 0.f, 0.f};
        for (int i = lane * 4; i < a.c_chunk; i += 256)
            asm volatile("ds_write_b128 %0, %1" ::"v"(lds_addr(colw_w) + (uint32_t)(i * 4)), "v"(zero4) : "memory");
        cleared = true;
    };

    for (; left > 0 && h < a.v_heads; at = 0, rb = (rb + 1 == a.c_nrb) ? 0 : rb + 1, h += (rb == 0)) {
        // the part of the row block's stages that belongs to the share
        int c0 = ck0, c_past = c1;  // its first key, and one past its last
        if constexpr (!ONE) {
            const int all = a.c_line.between(rb, cx * a.c_cs, (cx + 1) * a.c_cs);
            if (all <= 0) continue;  // no row of it sees the chunk
            const int first = max(0, at - a.c_line.start), past = max(0, min(all, at + min(left, 0x3fffffff) - a.c_line.start));
            left -= all + a.c_line.start - at;
            if (past <= first) break;  // the share ends with places for its start
            c0 += first * a.c_unit * KT;
            c_past = min(c1, ck0 + past * a.c_unit * KT);
        }
        const int row0 = rb * BLOCK_ROWS;                        // first query row of the unit
        // keys of these stages that some row of the unit sees
        int kend = c_past;
        if (a.causal) kend = min(kend, a.k_past + rows_past<FOLD>(a, row0 + BLOCK_ROWS));
        const int nst = (kend > c0) ? (kend - c0 + KT - 1) / KT : 0;
        if (nst == 0) {  // block-uniform
            if constexpr (ONE) break;
            else continue;
        }
        const int n_whole = (D == 64 || a.D == D) ? min(nst, (a.Sk - c0) / KT) : 0;  // stages inside the tensor, of rows as wide as compiled (64: or not)
        // REV: the stages that all rows of the block see are streamed backwards, [0, n_rev)
        const int n_rev = !REV ? 0 : plain_stages(c0, nst, a.causal ? min(a.k_past + rows_first<FOLD>(a, row0, BLOCK_ROWS), a.Sk - 1) : a.Sk - 1);
        auto pos = [&](int st) { return REV && st < n_rev ? n_rev - 1 - st : st; };
        if constexpr (!ONE) {  // what derives from these is formed anew, not kept from unit to unit
#pragma unroll
            for (int t = 0; t < NTA; ++t) asm volatile("" : "+v"(take[t]));
#pragma unroll
            for (int j = 0; j < IPW; ++j) asm volatile("" : "+v"(g_off[j]));
        }

        // ---- stationary operand: this wave's query rows of head h, as they are in memory
        const int qw0 = row0 + wave * ROWS_W;
        half8 qf[NB][NT];
        auto load_q_rows = [&]() {
            int lane_o = lane;
            asm volatile("" : "+v"(lane_o));  // addresses are formed here, not kept for a second call
            load_quads<D, NB, FOLD>(a, b, h, qw0, lane_o, qf);
        };
        auto take_q_rows = [&]() {  // once they have come
            int lane_o = lane;
            asm volatile("" : "+v"(lane_o));
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                quad_transpose(qf[nb]);
                if (a.D != D) zero_past_dim(qf[nb], a.D, lane_o >> 5);
            }
        };
        // the form the matrix pipe takes: pre-scaled (sign included), or raw with the scale's sign
        auto shape_q = [&](bool scaled) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    if (PRE && scaled) qf[nb][t] = prescale(qf[nb][t], a.negate ? -a.c : a.c);
                    else if (a.c == 0.f) qf[nb][t] = kZero8;
                    else if (a.negate) qf[nb][t] = flip_sign(qf[nb][t]);
                }
        };
        const char *kp = reinterpret_cast<const char *>(a.k + (int64_t)b * a.ks_b +
                                                        (int64_t)kv_head(h, a.kv_group, a.kv_magic) * a.ks_h);
        const int64_t k_row_b = a.ks_s * 2;

        // stage `st` of the unit into ring slot `slot`
        // The stages of a stream are requested in order; k_src is where the next one starts.
        const char *k_src;
        auto fetch_whole = [&](int slot) __attribute__((always_inline)) {  // such a stage
            char *dst = ring_w + slot * STAGE_BYTES;
            if (D != 64 || __builtin_expect(a.D == D, 1)) {
#pragma unroll
                for (int j = 0; j < IPW; ++j) dma16(k_src + g_off[j], dst + j * 1024);
            } else {
#pragma unroll
                for (int j = 0; j < IPW; ++j) dma16(g_off[j] == kPastDim ? reinterpret_cast<const char *>(g_zero_piece) : k_src + g_off[j], dst + j * 1024);
            }
            k_src += KT * k_row_b;
        };
        auto fetch_stage = [&](int st, int slot) __attribute__((always_inline)) {
            if (__builtin_expect(st < n_whole, 1)) {
                if (REV) k_src = kp + (int64_t)(c0 + pos(st) * KT) * k_row_b;
                fetch_whole(slot);
                return;
            }
            const int kb = c0 + pos(st) * KT;
            char *dst = ring_w + slot * STAGE_BYTES;
            if (D == 256 && kb + KT <= a.Sk) {  // narrower rows, as in the row pass (the smaller kernels are no faster with it)
                const char *base = kp + kb * k_row_b;
#pragma unroll
                for (int j = 0; j < IPW; ++j) dma16(g_off[j] == kPastDim ? reinterpret_cast<const char *>(g_zero_piece) : base + g_off[j], dst + j * 1024);
            } else {  // rows past the last key re-read it (the consumer masks them), pieces past the head dim are zeros
                int lane_o = lane;
                asm volatile("" : "+v"(lane_o));  // formed here, not kept in registers through the stream
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
        // Stage `st` of the stream [.., s1) is entered: the one behind it has landed (this wave's pieces; the barrier extends that
        // to everyone's), and every wave is done reading the stage before it, whose slot takes the next fetch.
        auto enter = [&](int st, int s1) __attribute__((always_inline)) {
            wait_stages<NS, IPW>(s1 - st);
            block_barrier();
        };
        auto fetch_ahead = [&](int st, int s1, int slot) __attribute__((always_inline)) {
            if (st + NS - 1 < s1) fetch_stage(st + NS - 1, slot);
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

        // ---- prologue of the unit's first phase: NS - 1 stages in flight, then the statistics, then the query rows, which
        // share their latency; the statistics are worked on while the query rows come
        auto fetch_first = [&](int s0, int s1) __attribute__((always_inline)) {
            k_src = kp + (int64_t)(c0 + s0 * KT) * k_row_b;
#pragma unroll
            for (int st = 0; st < NS - 1; ++st)
                if (s0 + st < s1) fetch_stage(s0 + st, st);
        };
        const int n_pre_most = PRE ? min(nst, max(0, (a.pre_end - c0) / KT)) : 0;
        fetch_first(0, nst);

        // ---- the row statistics that pass 1 left: (m, log2 l), or the parts' (m, l)
        const int qi = row0 + tid;
        const bool real = tid < BLOCK_ROWS && qi < a.v_rows;
        int parts = 1;
        const float2 *stat = a.stat;
        {
            const int rb1 = (row0 + wave * 64) / ROWS1;  // pass 1's row block (ROWS1 rows: those of a wave lie in one)
            const int i1 = (b * a.v_heads + h) * a.n_qblk + rb1;
            int w0 = 0;
            if (!a.r_whole) {
                const int start = (b * a.v_heads + h) * (int)a.r_by_head.d + a.r_line.places(rb1) + a.r_line.start;
                w0 = a.r_by_seg.quot(start);
                parts = a.r_by_seg.quot(start + a.r_line.n(rb1) - 1) - w0 + 1;
            }
            stat += ((int64_t)w0 + i1) * ROWS1 + (min(qi, a.v_rows - 1) - rb1 * ROWS1);
        }
        constexpr int PB = (NB == 1 && D < 256) ? 16 : D < 256 ? 8 : 4;  // parts in flight
        float2 part[PB];
        auto load_parts = [&](int ch0) {  // (past the last one: that one again, for nothing)
#pragma unroll
            for (int j = 0; j < PB; ++j) part[j] = stat[(int64_t)min(ch0 + j, parts - 1) * ROWS1];
        };
        if ((BLOCK_ROWS >= THREADS || wave * 64 < BLOCK_ROWS) && row0 + wave * 64 < a.v_rows) load_parts(0);
        load_q_rows();

        // ---- meanwhile: the accumulator slice of a new chunk; the per-row constants, merged over the parts of pass 1.  (Inline
        // assembly: the compiler could make ordinary LDS accesses wait for the DMA.)
        if (!cleared) clear_slice();
        {
            float nl = -INFINITY;  // a row that is not averaged: every p comes out as 2^-inf = 0
            float mm = 0.f, lg = 0.f;
            if (real) {
                // Added up in split order: bit-reproducible.  The usual parts are unstabilised (m = 0) or empty (both 0), and
                // the row's sum is the sum of theirs.
                float ll = 0.f;
                uint32_t stab = 0;  // a bit of any m
                auto add_parts = [&](int ch0) {
#pragma unroll
                    for (int j = 0; j < PB; ++j) {
                        ll += (ch0 + j < parts) ? part[j].y : 0.f;
                        stab |= __float_as_uint(part[j].x);
                    }
                };
                add_parts(0);
                for (int ch0 = PB; ch0 < parts; ch0 += PB) {
                    load_parts(ch0);
                    add_parts(ch0);
                }
                lg = a.r_whole ? part[0].y : fast_log2(ll);
                mm = part[0].x;
                if (__builtin_expect((stab & 0x7fffffffu) != 0 && !a.r_whole, 0)) {
                    // A split that pass 1 left unstabilised reports m = 0 and a sum of up to 2^110;
                    // next to a stabilised split its weight 2^((0 - m) * c) alone underflows although
                    // the product does not: the weights are applied as two square roots.
                    mm = kNegBig * 4.f;
                    ll = 0.f;
                    for (int ch = 0; ch < parts; ++ch) {
                        const float2 v = stat[(int64_t)ch * ROWS1];
                        if (v.y == 0.f) continue;  // empty
                        const float mn = fmaxf(mm, v.x);
                        const float wa = fast_exp2((mm - mn) * (0.5f * a.c)), wb = fast_exp2((v.x - mn) * (0.5f * a.c));
                        ll = (ll * wa) * wa + (v.y * wb) * wb;
                        mm = mn;
                    }
                    lg = fast_log2(ll);
                }
                // -lg / c: the reciprocal's quotient and one correction by its remainder
                const float q = lg * inv_c;
                nl = tiny ? 0.f : -fmaf(fmaf(-q, cmul, lg), inv_c, q);
            }
            // a stabilised row switches the whole unit, or its wave (kRedoHeads), to the two-constant form
            const int sh = (tiny || __builtin_amdgcn_ballot_w64(mm != 0.f) != 0) ? 1 : 0;
            asm volatile("ds_write_b32 %0, %1" ::"v"(lds_addr(shift_s) + (uint32_t)(wave * 4)), "v"(sh) : "memory");
            if (tid < BLOCK_ROWS) {
                const uint32_t at = (uint32_t)(tid * 4);
                const float np = (nl == -INFINITY) ? -INFINITY : -lg, cm = (nl == -INFINITY) ? -INFINITY : -mm;
                asm volatile("ds_write_b32 %0, %1" ::"v"(lds_addr(nl_s) + at), "v"(nl) : "memory");
                if (PRE) asm volatile("ds_write_b32 %0, %1" ::"v"(lds_addr(np_s) + at), "v"(np) : "memory");
                asm volatile("ds_write_b32 %0, %1" ::"v"(lds_addr(lg_s) + at), "v"(lg) : "memory");
                asm volatile("ds_write_b32 %0, %1" ::"v"(lds_addr(cm_s) + at), "v"(cm) : "memory");
            }
        }
        take_q_rows();
        wait_stages<NS, IPW>(nst);
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
        const int n_pre = (!PRE || shifted) ? 0 : n_pre_most;

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
                fetch_first(s0, s1);
                wait_stages<NS, IPW>(s1 - s0);
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
                    col_ad = lds_addr(colw_w) + (uint32_t)((kb_t - ck0 + na * 32 + n) * 4);
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
                    const int kb = c0 + pos(st) * KT;
                    const bool first = SLOT == 0 && st == s0;
                    if (!first) enter(st, s1);
                    if (NS == 3) fetch_ahead(st, s1, (SLOT + NS - 1) % NS);
#pragma unroll
                    for (int q = 0; q < TILES; ++q) {
                        const int na = q / NB, nb = q % NB;
                        if (nb == 0) frag_wait(kf);
                        acc[q & 1] = chain(nb);
                        asm volatile("" : "+v"(acc[0]), "+v"(acc[1]));  // the chain stays where it was written
                        // (a ring of four: the fetch, which has time, does not stand between the barrier and the chain)
                        if (NS > 3 && q == 0) fetch_ahead(st, s1, (SLOT + NS - 1) % NS);
                        if (nb == NB - 1) {  // this fragment's last chain has been issued: read back the next one
                            if (na == 0) take_frag(std::integral_constant<int, SLOT * STAGE_BYTES + 32 * ROW_BYTES>{}, kf);
                            else take_frag(std::integral_constant<int, ((SLOT + 1) % NS) * STAGE_BYTES>{}, kf);
                        }
                        // the tile before: in this stage, or the last one of the previous stage
                        const int p_kb = (q > 0) ? kb : REV ? c0 + pos(st - 1) * KT : kb - KT;
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
                drain_begin(c0 + pos(sp - 1) * KT, NA - 1, NB - 1);
                drain_plain(acc[(TILES - 1) & 1], NB - 1);
                drain_end(NB - 1);
            }

            // ---- the rest of the phase, in rolled loops (the ring slot is a run-time value): the stages on the diagonal or
            // past the last key as far as some row of the wave sees them, [sp, sv), then those that none of its rows sees
            const int sv = min(s1, max(sp, n_seen));
            int slot = (sp - s0) % NS;
            auto enter_stage = [&](int st) {
                if (st > s0) enter(st, s1);
                fetch_ahead(st, s1, (slot == 0) ? NS - 1 : slot - 1);
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
            block_sync();  // the ring (and nl_s) is reused by the next phase or unit
        };

        // (one call site per form, so that the code of each exists once)
        int raw0 = 0;  // first stage of the raw phase
        if (PRE && n_pre > 0) {
            shape_q(true);
            run_phase(std::integral_constant<int, kFormPrescaled>{}, 0, n_pre, true);
            raw0 = n_pre;
            if (raw0 < nst) {  // the unit's last stages (causal: keys that not every row sees)
                load_q_rows();
                take_q_rows();
            }
        }
        if (raw0 < nst) {
            shape_q(false);
            if (shifted) run_phase(std::integral_constant<int, kFormShifted>{}, 0, nst, true);
            else run_phase(std::integral_constant<int, kFormRaw>{}, raw0, nst, raw0 == 0);
        }
        if constexpr (ONE) break;
    }

    // ---- add the waves' slices in wave order and store
    if (!cleared) clear_slice();  // no row of any unit sees the keys
    block_sync();
    float *slab = a.partial + ((int64_t)share + (int64_t)b * a.c_nchunks + cx) * a.c_chunk;
    for (int i = tid; i < c1 - ck0; i += THREADS) {
        float v = colw[i];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) v += colw[w * CHUNK + i];
        if (!ONE && a.c_direct) {
            const int64_t o = (int64_t)b * a.Sk + ck0 + i;
            a.out[o] = v * a.inv_norm;
            if (a.out_h) a.out_h[o] = (_Float16)(v * a.inv_norm);
        } else {
            slab[i] = v;
        }
    }
    if (ONE || a.c_direct || left <= a.c_line.start) break;
    block_sync();  // the accumulators are cleared again
    h = rb = at = 0;
    // the next chunk that some row sees
    do {
        if (++cx == a.c_nchunks) {
            cx = 0;
            ++b;
        }
    } while (cx * a.c_cs >= a.c_line.last);
    }
}

// ------------------------------------------------------------------------------------
// pass 1 on the same machinery: row maximum and sum of exponentials of the row blocks that a share of the line touches
// ------------------------------------------------------------------------------------
// Same orientation and stream as the column pass (Q stationary, K through the LDS-DMA ring), but the
// exponentials are added up per ROW: register i of a lane keeps the running sum of its row over the
// lane's keys for the part of the row block that the share has, and the 32 key lanes are added once at its end, in
// registers (fcs_rowfold.h; through LDS it took 1.2 us and the space of a fourth ring slot at D 128).
// Common case: 2^(c * s) without max subtraction, exact while every row sum of the split stays inside
// [2^-80, 2^110); a block that leaves that range redoes its keys in two more sweeps (row maxima, then
// sums of 2^((s - m) * c), the maximum subtracted before the scale).  FOLD: only the waves that hold rows of a
// head with such a row redo, as when each head had a block of its own; the others take part in the fetches and barriers.
// One row of a call out of range (K 65536, 16 on 2 heads, Q 128, D 64: blocks of 512 rows laid end to end):
// 156 us, with none 105, with every wave of the block redoing 198, head by head 174.  Writes (m, log2 l) per row, or
// (m, l) per row and part when row blocks are cut; the column pass merges the parts.
// PRE: see the column pass.  The common sweep runs its stages below a.pre_end on Q * c rounded to fp16 (then the
// rest on the raw operand) and accepts row sums below 2^20 only; a block that leaves the range reloads the raw
// operand for its stabilised sweeps, all waves of it: the column pass then takes the raw operand for the whole unit.
template <int D, int NB, int WAVES, bool BF, bool PRE, bool FOLD, bool ONE>
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
    static_assert(IPW >= 1 && KT * PPR == IPW * THREADS, "a stage is a whole number of DMA instructions per wave");
    static_assert(NS >= 3 && NS <= 4, "ring depth");
    constexpr bool NARROW = D > 64 && !FOLD;  // stages of rows narrower than compiled have a path of their own
    __shared__ __attribute__((aligned(16))) char ring[NS * STAGE_BYTES];
    __shared__ __attribute__((aligned(16))) float mrow[BLOCK_ROWS];      // row maxima of the stabilised sweeps
    __shared__ int bad_s[WAVES];
    __shared__ int2 redo_s[kRedoHeads<PRE, FOLD> ? WAVES : 1];  // of such a wave: the rows that are redone, from .x to one before .y

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const float cmul = a.c;

    // ---- where this workgroup's share of the line starts: (batch entry, head), row block, stage
    fetch_args(a);
    const int share = xcd_contiguous((int)blockIdx.x, a.r_blocks);  // neighbours on the line run on one XCD
    int pos = ONE ? share : share * a.r_seg;
    int left = ONE ? 1 : min(a.r_seg, a.r_len - pos);  // places of the share that are still to do
    const int bh = a.r_by_head.quot(pos, pos);
    int bx = 0;
    if (ONE || a.r_line.step == 0) bx = a.r_by_block.quot(pos);
    else for (int sum = 0; pos >= (sum += a.r_line.n(bx) + a.r_line.start); ++bx) {}
    int at = pos - a.r_line.places(bx);  // place in the row block
    int h, b = a.by_heads.quot(bh, h);

    uint32_t g_off[IPW];
#pragma unroll
    for (int j = 0; j < IPW; ++j) {
        const int P = (wave * IPW + j) * 64 + lane;
        const int row = P / PPR, pos = P % PPR;
        const int piece = pos ^ row_swizzle<D>(row);
        g_off[j] = (!NARROW || piece * 8 < a.D) ? (uint32_t)row * (uint32_t)(a.ks_s * 2) + (uint32_t)(piece * 16) : kPastDim;
    }
    char *ring_w = ring + wave * (IPW * 1024);
    uint32_t take[NTA];
#pragma unroll
    for (int t = 0; t < NTA; ++t)
        take[t] = lds_addr(ring) + (uint32_t)(n * ROW_BYTES + ((piece_of<NTA>(t, g) ^ row_swizzle<D>(n)) * 16));

    // what derives from these is formed anew behind the call, not kept in registers from row block to row block or (the
    // rare sweeps' addresses) through the common sweep
    int lane_i = lane;
    auto form_anew = [&]() {
        asm volatile("" : "+v"(lane_i));
#pragma unroll
        for (int t = 0; t < NTA; ++t) asm volatile("" : "+v"(take[t]));
#pragma unroll
        for (int j = 0; j < IPW; ++j) asm volatile("" : "+v"(g_off[j]));
    };

    // ---- the row block at hand: which of its stages belong to the share
    const int64_t k_row_b = a.ks_s * 2;
    const int kp_eff = a.causal ? a.k_past : 0x3fffffff - a.Sq;
    int row0, qw0, kc0, nst, n_whole, n_plain, n_seen, n_pre;
    const char *kp;
    auto set_block = [&]() {
        const int first = ONE ? at : max(0, at - a.r_line.start), past = ONE ? at + 1 : min(a.r_line.n(bx), at + left - a.r_line.start);
        row0 = bx * BLOCK_ROWS;
        qw0 = row0 + wave * ROWS_W;
        // the keys of these stages, cut at the last key any of the block's rows may see
        kc0 = first * a.r_unit * KT;
        int kc1 = min(a.Sk, kc0 + (past - first) * a.r_unit * KT);
        if (a.causal) kc1 = min(kc1, a.k_past + rows_past<FOLD>(a, row0 + BLOCK_ROWS));
        nst = (kc1 > kc0) ? (kc1 - kc0 + KT - 1) / KT : 0;
        n_whole = (a.D == D) ? min(nst, (a.Sk - kc0) / KT) : 0;  // stages inside the tensor, of rows as wide as compiled
        // leading stages that run on the pre-scaled operand in the common sweep (block-uniform)
        n_pre = PRE ? min(nst, max(0, (a.pre_end - kc0) / KT)) : 0;
        const int thr_wave_min = a.causal ? min(a.k_past + rows_first<FOLD>(a, qw0, ROWS_W), a.Sk - 1) : a.Sk - 1;
        const int thr_wave_max = a.causal ? a.k_past + (FOLD ? a.q_rows : qw0 + ROWS_W) - 1 : a.Sk - 1;
        n_plain = plain_stages(kc0, nst, thr_wave_min);
        n_seen = seen_stages(kc0, nst, thr_wave_max);
        if (qw0 >= a.v_rows) n_plain = n_seen = 0;  // none of the wave's rows exists
        kp = reinterpret_cast<const char *>(a.k + (int64_t)b * a.ks_b + (int64_t)kv_head(h, a.kv_group, a.kv_magic) * a.ks_h);
    };

    half8 qf[NB][NT];
    auto load_q = [&]() {  // this wave's query rows
        int lane_o = lane;
        asm volatile("" : "+v"(lane_o));  // addresses are formed here, not kept for a second call
        load_quads<D, NB, FOLD>(a, b, h, qw0, lane_o, qf);
    };
    // the form the matrix pipe takes: pre-scaled (sign included), or raw with the scale's sign
    auto shape_q = [&](bool scaled) {
        int lane_o = lane;
        asm volatile("" : "+v"(lane_o));
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            quad_transpose(qf[nb]);
            if (a.D != D) zero_past_dim(qf[nb], a.D, lane_o >> 5);
        }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                if (PRE && scaled) qf[nb][t] = prescale(qf[nb][t], a.negate ? -a.c : a.c);
                else if (a.negate) qf[nb][t] = flip_sign(qf[nb][t]);
            }
    };

    // The stages of a stream are requested in order; k_src is where the next one starts.
    const char *k_src;
    auto fetch_whole = [&](int slot) __attribute__((always_inline)) {  // a stage inside the tensor, of rows as wide as compiled
        char *dst = ring_w + slot * STAGE_BYTES;
#pragma unroll
        for (int j = 0; j < IPW; ++j) dma16(k_src + g_off[j], dst + j * 1024);
        k_src += KT * k_row_b;
    };
    auto fetch_stage = [&](int st, int slot) __attribute__((always_inline)) {
        if (__builtin_expect(st < n_whole, 1)) {
            fetch_whole(slot);
            return;
        }
        const int kb = kc0 + st * KT;
        char *dst = ring_w + slot * STAGE_BYTES;
        // Narrower rows: zeros past their end, nothing but the base formed anew.  (Every piece's row and channel formed for each
        // stage: B 16, H 8, S 4096, D 96 584 us against 556, B 8, S 2048, D 200 245 against 207.  Not for rows laid end to end, whose
        // kernels are out of scalar registers: B 4, 32 on 8 heads, Q 64, K 8192, D 128 with the selection 60.3 -> 61.1.)
        if (NARROW && kb + KT <= a.Sk) {
            const char *base = kp + kb * k_row_b;
#pragma unroll
            for (int j = 0; j < IPW; ++j) dma16(g_off[j] == kPastDim ? reinterpret_cast<const char *>(g_zero_piece) : base + g_off[j], dst + j * 1024);
        } else {  // rows past the last key re-read it (the consumer masks them), pieces past the head dim are zeros
            int lane_o = lane;
            asm volatile("" : "+v"(lane_o));  // formed here, not kept in registers through the stream
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
    // Stage `st` of the stream [.., s1) is entered: the one behind it has landed (this wave's pieces; the barrier extends that
    // to everyone's), and every wave is done reading the stage before it, whose slot takes the next fetch.
    auto enter = [&](int st, int s1) __attribute__((always_inline)) {
        wait_stages<NS, IPW>(s1 - st);
        block_barrier();
    };
    auto fetch_ahead = [&](int st, int s1, int slot) __attribute__((always_inline)) {
        if (st + NS - 1 < s1) fetch_stage(st + NS - 1, slot);
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
    // A wave that is not `active` takes part in the fetches and barriers alone.  `fetched`: the first NS - 1 stages have been
    // requested already.
    auto fetch_first = [&](int s0, int s1) __attribute__((always_inline)) {
        k_src = kp + (int64_t)(kc0 + s0 * KT) * k_row_b;
#pragma unroll
        for (int st = 0; st < NS - 1; ++st)
            if (s0 + st < s1) fetch_stage(s0 + st, st);
    };
    auto sweep = [&](auto max_c, auto shift_c, auto scaled_c, const int s0, const int s1, const bool active, const bool fetched) {
        constexpr bool MAXOP = decltype(max_c)::value;
        constexpr bool SHIFT = decltype(shift_c)::value;
        constexpr bool SCALED = decltype(scaled_c)::value;
        static_assert(!SCALED || (PRE && !MAXOP && !SHIFT), "only the common sweep of the pre-scaled variant");
        constexpr int TILES = NA * NB;
        static_assert(NA == 2 && TILES % 2 == 0, "fragment offsets and the two alternating accumulators");
        if (s1 <= s0) return;  // block-uniform
        if (!fetched) fetch_first(s0, s1);
        wait_stages<NS, IPW>(s1 - s0);
        block_sync();
        const int n = lane_i & 31, g = lane_i >> 5;
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
                if (!first) enter(st, s1);
                if (NS == 3) fetch_ahead(st, s1, (SLOT + NS - 1) % NS);
#pragma unroll
                for (int q = 0; q < TILES; ++q) {
                    const int na = q / NB, nb = q % NB;
                    if (nb == 0) frag_wait(kf);
                    acc[q & 1] = chain(nb);
                    asm volatile("" : "+v"(acc[0]), "+v"(acc[1]));
                    if (NS > 3 && q == 0) fetch_ahead(st, s1, (SLOT + NS - 1) % NS);
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
            if (st > s0) enter(st, s1);
            fetch_ahead(st, s1, (slot == 0) ? NS - 1 : slot - 1);
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
        block_sync();  // the ring may be refilled by the next sweep
    };

    // ---- the row blocks that the share touches.  The next one's rows and first stages are requested as soon as the sweep
    // over this one has left the ring, ahead of its row sums.
    set_block();
    load_q();
    fetch_first(0, PRE && n_pre > 0 ? n_pre : nst);
    for (;;) {
        form_anew();
        if (nst == 0) block_sync();  // (in the place of the sweep's barriers: bad_s is written again)
        shape_q(n_pre > 0);
        // ---- common path: no max subtraction; the pre-scaled stages first, then the raw ones
        reset_rows(std::false_type{});
        if constexpr (PRE) {
            sweep(std::false_type{}, std::false_type{}, std::true_type{}, 0, n_pre, true, true);
            if (n_pre > 0 && n_pre < nst) {
                load_q();
                shape_q(false);
            }
        }
        sweep(std::false_type{}, std::false_type{}, std::false_type{}, n_pre, nst, true, n_pre == 0);

        const int c_b = b, c_h = h, c_bx = bx, c_at = at, c_left = left, c_kc0 = kc0, c_qw0 = qw0, c_nst = nst;
        const bool c_pre = n_pre > 0;
        left -= a.r_line.n(bx) + a.r_line.start - at;
        const bool more = !ONE && left > a.r_line.start;  // (not more than places for the next one's start: nothing to do there)
        if (more) {
            at = 0;
            if (++bx == a.n_qblk) {
                bx = 0;
                if (++h == a.v_heads) {
                    h = 0;
                    ++b;
                }
            }
            set_block();
            load_q();
            fetch_first(0, PRE && n_pre > 0 ? n_pre : nst);
        }

        // ---- row sums over the 32 key lanes, in registers: a lane is left with row `rw` of each fragment, like its neighbour
        const int lane_r = lane_i;
        const int rw = 16 * ((lane_r >> 4) & 1) + 8 * ((lane_r >> 3) & 1) + 4 * (lane_r >> 5) + 2 * ((lane_r >> 2) & 1) + ((lane_r >> 1) & 1);
        float lt[NB], m_row[NB];
        bool has[NB], out[NB], bad = false;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            lt[nb] = fold_lanes_sum(rs[nb], lane_r);
            const int v = c_qw0 + nb * 32 + rw, qi = rows_first<FOLD>(a, v, 1);
            const int thr = a.causal ? min(a.k_past + qi, a.Sk - 1) : a.Sk - 1;  // last key this row sees
            has[nb] = c_nst > 0 && c_kc0 <= thr && v < a.v_rows;
            // ceiling 2^110 rather than 2^120: up to 512 key splits of a row are added up by the column pass
            out[nb] = has[nb] && !(lt[nb] >= 8.2718061e-25f && lt[nb] < (c_pre ? kRowSumHiPre : 1.2980742e+33f));
            bad = bad || out[nb];
            m_row[nb] = 0.f;
            if (!has[nb]) lt[nb] = 0.f;  // an empty split
        }
        const bool wbad = __builtin_amdgcn_ballot_w64(bad) != 0;
        if constexpr (kRedoHeads<PRE, FOLD>) {
            if (wbad) {  // rows of the heads from the wave's first such row to its last
                int lo = 0x7fffffff, hi = -1;
#pragma unroll
                for (int nb = 0; nb < NB; ++nb)
                    if (out[nb]) {
                        lo = min(lo, nb * 32 + rw);
                        hi = max(hi, nb * 32 + rw);
                    }
#pragma unroll
                for (int m = 1; m < 64; m *= 2) {
                    lo = min(lo, __shfl_xor(lo, m));
                    hi = max(hi, __shfl_xor(hi, m));
                }
                const int from = fold_head(c_qw0 + lo, a.fold_magic) * a.q_rows;
                const int past = (fold_head(c_qw0 + hi, a.fold_magic) + 1) * a.q_rows;
                if (lane == 0) redo_s[wave] = int2{from, past};
            }
        }
        // (inline assembly: an ordinary LDS access would wait for the requested stages)
        {
            const int f = wbad ? 1 : 0;
            const uint32_t at = lds_addr(bad_s) + (uint32_t)(wave * 4);
            asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(f) : "memory");
            block_sync();
            int any = 0;
            const uint32_t from = lds_addr(bad_s) + (uint32_t)((lane % WAVES) * 4);
            asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(any) : "v"(from) : "memory");
            bad = __builtin_amdgcn_ballot_w64(any != 0) != 0;  // block-uniform
        }

        // ---- rare: row maxima first, then sums with the maximum subtracted before the scale
        if (bad) {
            const int n_b = b, n_h = h, n_bx = bx, n_at = at, n_left = left;
            b = c_b;
            h = c_h;
            bx = c_bx;
            at = c_at;
            left = c_left;
            form_anew();
            set_block();
            FCS_WAIT_VM(0);  // the next row block's stages: requested again below
            block_sync();
            bool redo = true;  // wave-uniform
            if constexpr (kRedoHeads<PRE, FOLD>) {
                redo = false;
                for (int w = 0; w < WAVES; ++w)
                    if (bad_s[w]) redo = redo || (redo_s[w].x < qw0 + ROWS_W && redo_s[w].y > qw0);
                redo = __builtin_amdgcn_readfirstlane(redo) != 0;
            }
            load_q();
            shape_q(false);
            reset_rows(std::true_type{});
            sweep(std::true_type{}, std::false_type{}, std::false_type{}, 0, nst, redo, false);
            float mx[NB];
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                mx[nb] = fold_lanes_max(rs[nb], lane_r);
                if (!has[nb]) mx[nb] = 0.f;  // no visible key in this split: every exponential is masked anyway
                mrow[wave * ROWS_W + nb * 32 + rw] = mx[nb];
            }
            __builtin_amdgcn_wave_barrier();
            const int g = lane_i >> 5;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int i = 0; i < 16; ++i) nmax[nb][i] = -mrow[wave * ROWS_W + nb * 32 + 8 * (i >> 2) + 4 * g + (i & 3)];
            reset_rows(std::false_type{});
            sweep(std::false_type{}, std::true_type{}, std::false_type{}, 0, nst, redo, false);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                const float ls = fold_lanes_sum(rs[nb], lane_r);
                if (!redo) continue;  // m = 0 and the sum of the common path stand
                m_row[nb] = mx[nb];  // (0 where the split is empty)
                lt[nb] = has[nb] ? ls : 0.f;
            }
            b = n_b;
            h = n_h;
            bx = n_bx;
            at = n_at;
            left = n_left;
            if (more) {
                set_block();
                load_q();
                fetch_first(0, PRE && n_pre > 0 ? n_pre : nst);
            }
        }

        // ---- store: one of the two lanes that hold a row
        if ((lane_r & 1) == 0) {
            const int64_t i = ((int64_t)c_b * a.v_heads + c_h) * a.n_qblk + c_bx;
            float2 *dst = a.stat + (a.r_whole ? i : i + share) * BLOCK_ROWS + wave * ROWS_W + rw;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) dst[nb * 32] = float2{m_row[nb], a.r_whole ? fast_log2(lt[nb]) : lt[nb]};
        }
        if (!more) break;
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
    const dim3 grid((unsigned)p.c_blocks);
    if constexpr (D == 64 && !BF) {
        if (stream_prescaled(p, a)) {
            if (p.c_one) hipLaunchKernelGGL((fcs_colstream_kernel<D, NB, WAVES, BF, true, FOLD, true>), grid, dim3(64 * WAVES), 0, st, a);
            else hipLaunchKernelGGL((fcs_colstream_kernel<D, NB, WAVES, BF, true, FOLD, false>), grid, dim3(64 * WAVES), 0, st, a);
            return hipGetLastError();
        }
    }
    if (p.c_one) hipLaunchKernelGGL((fcs_colstream_kernel<D, NB, WAVES, BF, false, FOLD, true>), grid, dim3(64 * WAVES), 0, st, a);
    else hipLaunchKernelGGL((fcs_colstream_kernel<D, NB, WAVES, BF, false, FOLD, false>), grid, dim3(64 * WAVES), 0, st, a);
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
    const dim3 grid((unsigned)p.r_blocks);
    if constexpr (D == 64 && !BF) {
        if (stream_prescaled(p, a)) {
            if (p.r_one) hipLaunchKernelGGL((fcs_rowstream_kernel<D, NB, WAVES, BF, true, FOLD, true>), grid, dim3(64 * WAVES), 0, st, a);
            else hipLaunchKernelGGL((fcs_rowstream_kernel<D, NB, WAVES, BF, true, FOLD, false>), grid, dim3(64 * WAVES), 0, st, a);
            return hipGetLastError();
        }
    }
    if (p.r_one) hipLaunchKernelGGL((fcs_rowstream_kernel<D, NB, WAVES, BF, false, FOLD, true>), grid, dim3(64 * WAVES), 0, st, a);
    else hipLaunchKernelGGL((fcs_rowstream_kernel<D, NB, WAVES, BF, false, FOLD, false>), grid, dim3(64 * WAVES), 0, st, a);
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
