// Attention column means on gfx950 (MI355X): single-pass path with 64 query rows x up to 128 keys per wave, where the waves of
// fcs_fused.hip own 32 rows x up to 256.  Calls of up to 1024 keys: non-causal ones of heads of 65 .. 128 channels, and of up to 64
// with four key tiles per wave whose operand is not pre-scaled; causal ones.  Beyond 1024 keys (up to 2048) causal calls, and others of
// 65 .. 128 channels, have 32 rows per wave and five to eight key tiles (make_plan says where, with both sides' times): what
// they gain on fcs_fused.hip is the shared query rows and the four items that stay in the ring.
//
// Causal calls: a key tile behind the last key that any of 32 rows sees has no exponents, one on the diagonal is masked after them.  (Its
// MFMAs run all the same: a branch around a chain made the register allocator spill 400 registers.)
//
// What bounds the 32-row tile at 128 channels is moving operands, not arithmetic: every wave brings its own copy of its keys,
// so that a row block of 64 rows x 1024 keys of 128 channels takes 576 KB through the L2 -> LDS path (about 65 B/clk
// per compute unit: 8.9 k cycles of the 15.5 k that the block took at B 8, H 16, S 1024) and as much through the LDS read port.
// With 64 rows to a wave
//   * no key tile is fetched twice by a workgroup (eight key groups, one group of rows), and an operand fragment that has been read
//     back serves two MFMA chains: half of both streams;
//   * the 64 query rows come once per workgroup, by DMA into an LDS tile that all waves read;
//   * the ring's last three items stay for the next row block of the same key head, which walks them in the opposite order; of 64-wide
//     heads all of them stay, and a key head is fetched once per workgroup.
// B 8 H 16 S 1024 D 128 bf16 60.1 -> 47.2 us per call.  What is left there: without the key fetches it would be 7 % faster,
// without three of four MFMAs 14 %, without phase 3 5 %.  64-wide heads are bound by the exponents either way: bf16 B 64 H 16 S 1024
// 256.9 -> 239.7.  (Their pre-scaled operand was tried: 245 -> 231 at B 64, 2 .. 13 % slower with two and three tiles per wave, and
// the rows' way through registers cannot be expressed safely in a loop with two waits; not built.)
//
// The scores of a wave (2 x 4 tiles) fill 128 registers as there, both chunks of 64 channels of wide query rows 64, two half tiles of
// keys 32.  A tile's exponents run under the next tile's MFMAs, a 32-row fragment under each chunk's.  (All tiles' first chunks, then all
// second ones, with one chunk of the rows in registers at a time, has MFMAs alone in its first half: S 1024 D 96 52.0 against
// 49.5 us, D 128 52.5 against 51.8, S 1300 D 128 113.3 against 109.1.)  What makes room: the row sums are added up behind
// phase 1 (running sums would be 32 registers more; they spilled, or were 4 % slower), and the rare path is marked as such,
// since the register allocator otherwise spilled a tile's exponentials to spare it (67 us at B 8, H 16, S 1024, D 128).
//
// The rest is fcs_fused.hip's: e = 2^(c s) without max subtraction while every row sum lands in [2^-80, 2^120), in-lane
// column sums, one barrier per row block, a slab of column sums per workgroup; a row block outside the range is redone
// with the row maxima subtracted.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <stdio.h>

#include "fcs_device.h"
#include "fcs_kernels.h"
#include "fcs_rowfold.h"

namespace fcs {

namespace {

constexpr float kSumLo = 8.2718061e-25f;  // 2^-80
constexpr float kSumHi = 1.3292280e+36f;  // 2^120

__device__ __attribute__((aligned(16))) unsigned int g_tall_zeros[4];  // the pieces of query rows past the head dim

#define FCS_WAIT_VM(N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory")
#define FCS_OPAQUE_V(x) asm volatile("" : "+v"(x))

__device__ __forceinline__ void pin16(float (&v)[16])
{
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]), "+v"(v[8]), "+v"(v[9]),
                 "+v"(v[10]), "+v"(v[11]), "+v"(v[12]), "+v"(v[13]), "+v"(v[14]), "+v"(v[15]));
}

// Four operand pieces of a row from LDS: those at `at`, and 2, 4 and 6 pieces on (the swizzles below only exchange bits of
// the piece number).  Only issued here: take_wait stands between this and the first use.  (Inline assembly: the
// compiler would make an ordinary LDS read wait for all DMA.)
template <int OFF>
__device__ __forceinline__ void take_issue(uint32_t at, half8 (&dst)[4])
{
    const uint32_t a1 = at ^ 32u, a2 = at ^ 64u, a3 = at ^ 96u;
    asm volatile("ds_read_b128 %0, %4 offset:%8\n\tds_read_b128 %1, %5 offset:%8\n\tds_read_b128 %2, %6 offset:%8\n\tds_read_b128 %3, %7 offset:%8"
                 : "=&v"(dst[0]), "=&v"(dst[1]), "=&v"(dst[2]), "=&v"(dst[3])
                 : "v"(at), "v"(a1), "v"(a2), "v"(a3), "n"(OFF)
                 : "memory");
}
__device__ __forceinline__ void take_wait(half8 (&dst)[4])
{
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(dst[0]), "+v"(dst[1]), "+v"(dst[2]), "+v"(dst[3])::"memory");
}

// this lane's number, from no register
__device__ __forceinline__ int lane_number()
{
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}
// both at once, where nothing is to be done in between
__device__ __forceinline__ void take_now(uint32_t at, half8 (&dst)[4])
{
    const uint32_t a1 = at ^ 32u, a2 = at ^ 64u, a3 = at ^ 96u;
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\tds_read_b128 %3, %7\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(dst[0]), "=&v"(dst[1]), "=&v"(dst[2]), "=&v"(dst[3])
                 : "v"(at), "v"(a1), "v"(a2), "v"(a3)
                 : "memory");
}

}  // namespace

// DC: chunks of 64 channels.  NB: 32-row fragments per wave.  TPW: 32-key tiles per wave.  NARROW: the head dim is less than DC x 64.
template <int DC, int NB, int TPW, bool BF, bool NARROW, bool CAUSAL>
__global__ __launch_bounds__(512, 2) void fcs_tall_kernel(const Args a)
{
    constexpr int ROWS = 32 * NB;
    constexpr int NT = 4;                // MFMA steps per chunk of 64 channels
    constexpr int STEPS = DC * TPW;      // ring items of a row block: (half) tiles, 32 keys x 64 channels; the chunks of a tile one after the other
    constexpr bool KEEP_ALL = DC == 1 && NB == 2;   // every item of a key head stays in the ring
    constexpr int NS = KEEP_ALL ? TPW : NB == 2 ? 3 : 4;              // ring slots per wave; item j of every row block lives in slot j % NS
    constexpr int ITEM = 4096;
    constexpr int QROW = DC * 128, QTILE = ROWS * QROW, QI = (DC * NB + 1) / 2;  // QI: a wave's DMA instructions for its 8 query rows
    static_assert(KEEP_ALL || STEPS > NS, "the waits below count on a request at the first step");
    __shared__ __attribute__((aligned(256))) char ring[8 * NS * ITEM];
    __shared__ __attribute__((aligned(256))) char qtile[2 * QTILE];  // the unit's query rows, double-buffered
    __shared__ __attribute__((aligned(16))) float part[2 * ROWS * 8];  // row sums per (row, wave), double-buffered
    __shared__ __attribute__((aligned(16))) float wv[8 * ROWS];        // per wave: a value per row

    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, g = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int hgi, b, qwg;
    {
        int bx, by, bz;
        xcd_contiguous_block(bx, by, bz);
        qwg = bx % a.f_nwgq;
        b = bx / a.f_nwgq;
        hgi = by;
    }
    // the walk over units (head, row block of ROWS rows), row blocks innermost
    const int h_begin = hgi * a.f_hpg, n_heads = min(a.H, h_begin + a.f_hpg) - h_begin;
    const int rb_first = qwg * a.f_rbpw;
    // Causal row blocks see more and more keys: a workgroup takes every f_nwgq-th of them, there and back, so that all have alike.
    auto row_block = [&](int r) { return !CAUSAL ? rb_first + r : (r & 1) ? (r + 1) * a.f_nwgq - 1 - qwg : r * a.f_nwgq + qwg; };
    const int rb_n = CAUSAL ? a.f_rbpw - (row_block(a.f_rbpw - 1) >= a.f_nqblk ? 1 : 0) : min(a.f_rbpw, a.f_nqblk - rb_first);
    const int n_units = rb_n * n_heads;
    // key tile t of the wave holds keys [kbase + kstep t, ..), moved back to end at the last key where it would reach past it; its
    // columns then repeat keys of the tile before and count for nothing: those of a lane are t > tmax_lane.  Causal calls deal the
    // tiles to the waves in turn, so that the keys that a row block sees are spread over all of them.
    const int kbase = CAUSAL ? wave * 32 : wave * TPW * 32;
    constexpr int kstep = CAUSAL ? 256 : 32;
    auto tile_first = [&](int t) { return min(kbase + t * kstep, a.Sk - 32); };
    auto tiles_counted = [&](int l) { return (l + a.Sk - 32 - kbase) >> (CAUSAL ? 8 : 5); };  // arithmetic shift: floor, also when negative
    const int tmax_lane = tiles_counted(n);

    const int64_t q_row_b = a.qs_s * 2;  // (of either sign, as on the two-pass path)
    const uint32_t k_row_b = (uint32_t)a.ks_s * 2u;
    const char *q_batch = reinterpret_cast<const char *>(a.q + (int64_t)b * a.qs_b);
    const char *k_batch = reinterpret_cast<const char *>(a.k + (int64_t)b * a.ks_b);
    const int64_t q_head_b = a.qs_h * 2, k_head_b = a.ks_h * 2;
    char *my_ring = ring + wave * (NS * ITEM);

    // ---- DMA.  A key item is 32 rows x 128 bytes; an instruction brings 8 rows, lane L piece (16 bytes) L % 8 of row L / 8,
    // stored XOR-swizzled (position p of row r holds piece p ^ ((r >> 1) & 7)).  Instructions 0 and 2, and 1 and 3, have the same
    // lane offsets, 16 rows apart.
    uint32_t k_voff[2], k_voff_n[NARROW ? 2 : 1];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t piece_b = (uint32_t)(((lane & 7) ^ ((i * 4 + (lane >> 4)) & 7)) * 16);
        const uint32_t row = (uint32_t)((lane >> 3) + 8 * i) * k_row_b;
        k_voff[i] = row + piece_b;
        // (second chunk of a narrower head: a piece past the head dim is replaced by the row's first of the chunk; the query
        // rows hold zeros there)
        if (NARROW) k_voff_n[i % (NARROW ? 2 : 1)] = row + ((int)((DC - 1) * 64 + (piece_b >> 1)) < a.D ? piece_b : 0u);
    }
    auto dma = [](const char *src, char *dst) {
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src, (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
    };
    auto fetch_item = [&](int64_t head_b, int tile, int chunk, int slot) {
        const char *src = k_batch + head_b + (size_t)tile_first(tile) * k_row_b + chunk * 128;
        char *dst = my_ring + slot * ITEM;
        FCS_OPAQUE_V(k_voff[0]);
        FCS_OPAQUE_V(k_voff[1]);
        const char *src2 = src + (size_t)(16 * k_row_b);
        if (NARROW) {
            const bool last = chunk == DC - 1;
            const uint32_t v0 = last ? k_voff_n[0] : k_voff[0], v1 = last ? k_voff_n[NARROW ? 1 : 0] : k_voff[1];
            dma(src + v0, dst);
            dma(src + v1, dst + 1024);
            dma(src2 + v0, dst + 2048);
            dma(src2 + v1, dst + 3072);
        } else {
            dma(src + k_voff[0], dst);
            dma(src + k_voff[1], dst + 1024);
            dma(src2 + k_voff[0], dst + 2048);
            dma(src2 + k_voff[1], dst + 3072);
        }
    };
    // the wave's eighth of a unit's query rows: 4 rows x 256 bytes per instruction, position p of row r holds piece p ^ (r & 15) (one
    // chunk: 8 rows x 128 bytes, as a key item);
    // rows past the last averaged one repeat it (they are given no weight, which would not do for a NaN in a row that is not averaged)
    auto fetch_q = [&](int head, int row0, int buf) {
        const char *slice = q_batch + (int64_t)head * q_head_b;
        // (32 rows of one chunk are four instructions: the waves 4 .. 7 bring what 0 .. 3 do, so that all count the same)
        const int w = DC * NB == 1 ? wave & 3 : wave;
        constexpr int RI = 1024 / QROW;  // rows of an instruction
        char *dst = qtile + buf * QTILE + w * (QI * 1024);
        int l = lane;
        FCS_OPAQUE_V(l);
#pragma unroll
        for (int i = 0; i < QI; ++i) {
            const int r = (w * QI + i) * RI + (DC == 2 ? l >> 4 : l >> 3);
            const int piece = DC == 2 ? (l & 15) ^ (r & 15) : (l & 7) ^ ((r >> 1) & 7);
            const char *src = slice + min(row0 + r, a.q_rows - 1) * q_row_b + piece * 16;
            if (NARROW && piece * 8 >= a.D) src = reinterpret_cast<const char *>(g_tall_zeros);
            dma(src, dst + i * 1024);
        }
    };

    // ---- read-back.  Lane (n, g) takes, for step tt of a chunk, piece 2 tt + g of row n.
    uint32_t k_take = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)my_ring + (uint32_t)(n * 128 + ((g ^ ((n >> 1) & 7)) * 16));
    uint32_t q_take = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)qtile + (DC == 2 ? (uint32_t)(n * 256 + ((n >> 3) & 1) * 128 + ((g ^ (n & 7)) * 16)) : (uint32_t)(n * 128 + ((g ^ ((n >> 1) & 7)) * 16)));

    float col_acc[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) col_acc[t] = 0.f;
    float *wv_w = wv + wave * ROWS;

    // Two orders of the items alternate between the row blocks of a key head: 0 .. STEPS-1 and (rot) back.  Item j is chunk j % DC of key
    // tile j / DC; the scores of step s are in acc[.][s / DC], which is tile s / DC or (rot) TPW - 1 - s / DC.
    int rot = 0;
    auto slot_of = [&](int s) { return rot ? (STEPS - 1 - s) % NS : s % NS; };
    auto tile_of = [&](int s) { return rot ? TPW - 1 - s / DC : s / DC; };  // of step s
    auto chunk_of = [&](int s) { return rot ? DC - 1 - s % DC : s % DC; };
    auto tile_at = [&](int t) { return rot ? TPW - 1 - t : t; };  // of accumulator t

    int cur_rb = 0, cur_hr = 0;  // row block and head of the current unit, relative
    auto key_off = [&](int hr) { return (int64_t)kv_head(h_begin + hr, a.kv_group, a.kv_magic) * k_head_b; };
    int64_t k_cur = key_off(0);

    fetch_q(h_begin, row_block(0) * ROWS, 0);
#pragma unroll
    for (int s = 0; s < NS; ++s) fetch_item(k_cur, s / DC, s % DC, s);
    FCS_WAIT_VM(0);
    __syncthreads();

    // the scale with its sign (a score of negated query rows, times c, has the very bits of the score times -c); scalar
    const float cs = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, a.negate ? -a.c : a.c)));
    for (int unit = 0; unit < n_units; ++unit) {
        const int h = h_begin + cur_hr, row0 = row_block(cur_rb) * ROWS;
        // the next unit (the last one is followed by itself)
        int nxt_rb = cur_rb, nxt_hr = cur_hr;
        if (unit + 1 < n_units && ++nxt_rb == rb_n) {
            nxt_rb = 0;
            ++nxt_hr;
        }
        const int64_t k_nxt = key_off(nxt_hr);
        const int next_key_head = __builtin_amdgcn_readfirstlane(k_nxt != k_cur ? 1 : 0);

        // The query rows are in their tile since the barrier before.  The first NS key items are in the ring: left behind by the
        // unit before, or requested during its last steps.
        half8 qf[DC][NB][NT], kf[2][NT];  // [chunk][32-row fragment]
        FCS_OPAQUE_V(q_take);
        FCS_OPAQUE_V(k_take);
        const uint32_t q_at = q_take + (uint32_t)((unit & 1) * QTILE);
#pragma unroll
        for (int dc = 0; dc < DC; ++dc) {
            take_issue<0>(q_at ^ (uint32_t)(chunk_of(dc) * 128), qf[dc][0]);
            if constexpr (NB == 2) take_issue<32 * QROW>(q_at ^ (uint32_t)(chunk_of(dc) * 128), qf[dc][NB - 1]);
        }
        FCS_WAIT_VM(0);
        take_issue<0>(k_take + (uint32_t)(slot_of(0) * ITEM), kf[0]);

        floatx16 acc[NB][TPW];
        float e[NB][TPW][16];
        // causal: the last key that all / any of 32 rows see; a tile behind the latter has no products and no exponents
        auto seen_by_all = [&](int nb) { return a.k_past + row0 + nb * 32; };
        auto hidden = [&](int nb, int t) { return CAUSAL && tile_first(tile_at(t)) > seen_by_all(nb) + 31; };
        auto exp_tile = [&](int nb, int t) {  // e = 2^(c s); a column that does not count, a key that the row does not see: 2^-inf
            const float bias = tile_at(t) <= tmax_lane ? 0.f : -INFINITY;
            const int key0 = tile_first(tile_at(t));
#pragma unroll
            for (int i = 0; i < 16; ++i) e[nb][t][i] = acc[nb][t][i];
            if (!hidden(nb, t)) {
#pragma unroll
                for (int i = 0; i < 16; ++i) e[nb][t][i] = fast_exp2(fmaf(e[nb][t][i], cs, bias));
            }
            if (CAUSAL && key0 + 31 > seen_by_all(nb)) {  // (in place, and one-sided: else both sides' registers are live)
                pin16(e[nb][t]);
                int rel = key0 + n - seen_by_all(nb) - 4 * g;  // seen by the row of register i: rel <= 8 (i / 4) + i % 4
                FCS_OPAQUE_V(rel);
#pragma unroll
                for (int i = 0; i < 16; ++i) e[nb][t][i] = rel <= 8 * (i >> 2) + (i & 3) ? e[nb][t][i] : 0.f;
            }
            pin16(e[nb][t]);  // (else the exponents sink below the last MFMA)
        };

        // ---------------- phase 1
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const int dc = s % DC, t = s / DC;
            // (the two waves of a SIMD take turns at the higher priority, as in fcs_fused.hip)
            if (((s & 1) != 0) == (wave >= 4)) asm volatile("s_setprio 2");
            else asm volatile("s_setprio 0");
            if (s == 0) {
#pragma unroll
                for (int dc = 0; dc < DC; ++dc) {
                    take_wait(qf[dc][0]);
                    if constexpr (NB == 2) take_wait(qf[dc][NB - 1]);
                }
            }
            FCS_OPAQUE_V(k_take);  // addresses are formed where they are used
            take_wait(kf[s & 1]);
            if (s == 0) fetch_q(h_begin + nxt_hr, row_block(nxt_rb) * ROWS, (unit + 1) & 1);
            // the slot is free: it takes the item of step s + NS, or the next key head's item that belongs in it
            if (s + NS < STEPS) fetch_item(k_cur, tile_of(s + NS), chunk_of(s + NS), slot_of(s));
            else if (next_key_head) fetch_item(k_nxt, slot_of(s) / DC, slot_of(s) % DC, slot_of(s));
            // Item s + 1 has landed once at most the items requested behind it are outstanding (step s + 1 - NS requested it; the
            // last step that requests one of this unit is STEPS - NS - 1).  The query rows, requested before all of them, have too.
            if (!KEEP_ALL && s + 1 >= NS && s + 1 < STEPS) FCS_WAIT_VM((STEPS - 2 - s < NS - 1 ? STEPS - 2 - s : NS - 1) * NT);
            if (s + 1 < STEPS) take_issue<0>(k_take + (uint32_t)(slot_of(s + 1) * ITEM), kf[(s + 1) & 1]);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                floatx16 c = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
                if (dc) c = acc[nb][t];
#pragma unroll
                for (int tt = 0; tt < NT; ++tt) c = mfma16<BF>(qf[dc][nb][tt], kf[s & 1][tt], c);
                acc[nb][t] = c;
            }
            if (t > 0) {  // VALU work of the tile before under this one's MFMAs, spread over its steps
                if (dc == 0) exp_tile(0, t - 1);
                if (NB == 2 && dc == DC - 1) exp_tile(NB - 1, t - 1);
            }
        }
        exp_tile(0, TPW - 1);
        if (NB == 2) exp_tile(NB - 1, TPW - 1);

        if (KEEP_ALL) {  // the next unit's query rows have landed: behind them is the next key head, or nothing
            if (next_key_head) FCS_WAIT_VM(STEPS * NT);
            else FCS_WAIT_VM(0);
        }

        // ---------------- row sums over lanes and waves: one barrier, which also publishes the next unit's query rows
        float *pt = part + (unit & 1) * (ROWS * 8);
        // the row (of 32) whose total over this wave's keys a lane is left with, like its neighbour
        int lane_r = lane;
        FCS_OPAQUE_V(lane_r);  // addresses are formed here, not kept through phase 1
        const int g_r = lane_r >> 5;
        const int row_w = 16 * ((lane_r >> 4) & 1) + 8 * ((lane_r >> 3) & 1) + 4 * g_r + 2 * ((lane_r >> 2) & 1) + ((lane_r >> 1) & 1);
        auto fold_rows = [&](int nb, float v) {
            if ((lane_r & 1) == 0) pt[(nb * 32 + row_w) * 8 + wave] = v;
        };
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            float rs[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                rs[i] = e[nb][0][i] + e[nb][1][i];
#pragma unroll
                for (int t = 2; t + 1 < TPW; t += 2) rs[i] += e[nb][t][i] + e[nb][t + 1][i];
                if (TPW % 2) rs[i] += e[nb][TPW - 1][i];
            }
            fold_rows(nb, fold_lanes_sum(rs, lane_r));
        }
        __syncthreads();
        // lane L adds up row L (32 rows: the upper half-wave does what the lower does); every wave sees all of the rows' parts
        bool slow;
        {
            const int row = lane_r & (ROWS - 1);
            const floatx4 f0 = *reinterpret_cast<const floatx4 *>(pt + row * 8), f1 = *reinterpret_cast<const floatx4 *>(pt + row * 8 + 4);
            const float tot = ((f0[0] + f0[1]) + (f0[2] + f0[3])) + ((f1[0] + f1[1]) + (f1[2] + f1[3]));
            bool ok = true;
            float most = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                ok = ok && f0[j] < kSumHi && f1[j] < kSumHi;  // false for NaN
                most = fmaxf(most, fmaxf(f0[j], f1[j]));
            }
            slow = __builtin_amdgcn_ballot_w64(!ok || !(most >= kSumLo)) != 0;
            wv_w[row] = (row0 + row < a.q_rows) ? __builtin_amdgcn_rcpf(tot) : 0.f;
            __builtin_amdgcn_wave_barrier();
        }

        if (__builtin_expect(!slow, 1)) {
            // ---------------- phase 3: column sums of e * w, this row block's by themselves first
            float sum[TPW];
#pragma unroll
            for (int t = 0; t < TPW; ++t) sum[t] = 0.f;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int i4 = 0; i4 < 4; ++i4) {
                    const floatx4 w4 = *reinterpret_cast<const floatx4 *>(wv_w + nb * 32 + 8 * i4 + 4 * g_r);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int t = 0; t < TPW; ++t) sum[t] = fmaf(e[nb][t][4 * i4 + j], w4[j], sum[t]);
                }
#pragma unroll
            for (int t = 0; t < TPW; ++t) col_acc[t] += rot ? sum[TPW - 1 - t] : sum[t];
        } else {
            // ------------ rare: the softmax with the row maximum subtracted, 32 rows after the other, two sweeps over the keys that the
            // block sees with one score tile in registers at a time: row maxima and sums, then column sums.  The keys come through the
            // ring as in phase 1; what the ring held for the next unit is requested again behind the sweeps.
            // What bounds it is VALU work, up to 22 instructions a score, and that all of a unit's waves go through it for one row.  us per
            // call with every row out of range, of scores formed three times over from ordinary loads (64 lanes to 32 rows), this, and
            // the kernel that served the call before: causal H 32 S 1000 D 128 194, 66, 53; Q 128 K 2048 73, 35, 31; H 24 S 2048 393, 125,
            // 97; H 32 S 1500 D 64 160, 76, 64; B 8 H 16 S 1024 D 128 541, 227, 425, S 1000 D 96 435, 240, 260, S 1800 D 96 1114, 898, 505.
            // With a hundredth of the rows so it is the quickest of the three but for Q 128 K 2048 (72, 34, 31).
            // From an opaque copy of the lane id: nothing of this is kept by the common path.
            int lane_s = lane;
            FCS_OPAQUE_V(lane_s);
            const int n_s = lane_s & 31, g_s = lane_s >> 5;
            const int seen_by_last = a.k_past + a.q_rows - 1;  // causal: rows past the averaged ones see what the last of those sees
            // the wave's tiles that any row of the block sees
            const int past = CAUSAL ? min(a.Sk, min(a.k_past + row0 + ROWS - 1, seen_by_last) + 1) : a.Sk;
            const int tiles = past > kbase ? min(TPW, (past - kbase + kstep - 1) / kstep) : 0, n_items = DC * tiles;
            const bool gone = !KEEP_ALL || next_key_head;  // the ring does not hold all of this key head
            FCS_WAIT_VM(0);
            if (KEEP_ALL && gone) {
#pragma unroll
                for (int s = 0; s < STEPS; ++s) fetch_item(k_cur, s, 0, s);
                FCS_WAIT_VM(0);
            }
            // The query rows are kept, or where registers do not suffice read again for each tile (what a loop spills costs more: a
            // reload waits for all fetches).
            constexpr bool KEEP_Q = NB * TPW < (DC == 2 ? 6 : CAUSAL ? 8 : 9);
            auto take_rows = [&](int nb, int dc, half8 (&q)[NT]) __attribute__((always_inline)) {
                take_now((q_at ^ (uint32_t)(dc * 128)) + (uint32_t)(nb * 32 * QROW), q);
#pragma unroll
                for (int tt = 0; tt < NT; ++tt) q[tt] = a.negate ? flip_sign(q[tt]) : q[tt];
            };
            // f(t, the scores of tile t, which of them count), for all of them
            auto sweep = [&](int nb, half8 (&qs)[DC][NT], auto f) __attribute__((always_inline)) {
                if (tiles == 0) return;
                if (!KEEP_ALL) {
                    FCS_WAIT_VM(0);
#pragma unroll
                    for (int j = 0; j < NS; ++j) fetch_item(k_cur, min(j, n_items - 1) / DC, min(j, n_items - 1) % DC, j);
                }
                int slot = 0;
#pragma unroll 1
                for (int t = 0; t < tiles; ++t) {
                    floatx16 c = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int dc = 0; dc < DC; ++dc) {
                        half8 kv[NT];
                        if (!KEEP_Q) take_rows(nb, dc, qs[dc]);
                        if (!KEEP_ALL) FCS_WAIT_VM((NS - 1) * NT);
                        take_now(k_take + (uint32_t)(slot * ITEM), kv);
                        if (!KEEP_ALL) {
                            const int ahead = min(DC * t + dc + NS, n_items - 1);  // (the last one again at the end: the waits count on a request)
                            fetch_item(k_cur, ahead / DC, ahead % DC, slot);
                        }
                        slot = slot + 1 == NS ? 0 : slot + 1;
#pragma unroll
                        for (int tt = 0; tt < NT; ++tt) {
                            // (the pieces past the head dim repeat others: an infinity there, times 0)
                            if (NARROW && dc == DC - 1 && dc * 64 + tt * 16 + (lane_number() >> 5) * 8 >= a.D) kv[tt] = kZero8;
                            c = mfma16<BF>(qs[dc][tt], kv[tt], c);
                        }
                    }
                    const int first = kbase + t * kstep;
                    if (first <= a.Sk - 32 && (!CAUSAL || first + 31 <= min(seen_by_all(nb), seen_by_last))) {
                        f(t, c, [](int) { return true; });
                    } else {
                        // the row of register i, 8 (i / 4) + 4 g + i % 4 of the 32, counts this lane's key: rel <= 8 (i / 4) + i % 4
                        // (from the lane number formed anew: a register that is kept for it is spilled, and a reload waits for all fetches)
                        const int lane_t = lane_number(), n_t = lane_t & 31, key = tile_first(t) + n_t;
                        const int rel = t > tiles_counted(n_t) || (CAUSAL && key > seen_by_last) ? 1 << 20 : CAUSAL ? key - seen_by_all(nb) - 4 * (lane_t >> 5) : -1;
                        f(t, c, [rel](int i) { return rel <= 8 * (i >> 2) + (i & 3); });
                    }
                }
            };
#pragma unroll 1
            for (int nb = 0; nb < NB; ++nb) {
                half8 qs[DC][NT];
#pragma unroll
                for (int dc = 0; dc < DC; ++dc)
                    if (KEEP_Q) take_rows(nb, dc, qs[dc]);
                // row values over lanes and waves: f(the 8 waves' parts of a row) goes to wv_w, and from there to v.  The barrier in
                // front is for the part buffer's last readers.
                const int row = nb * 32 + n_s;
                auto reduce = [&](float mine, float (&v)[16], auto f) {
                    __syncthreads();
                    const int rw = 16 * ((lane_s >> 4) & 1) + 8 * ((lane_s >> 3) & 1) + 4 * g_s + 2 * ((lane_s >> 2) & 1) + ((lane_s >> 1) & 1);
                    if ((lane_s & 1) == 0) pt[(nb * 32 + rw) * 8 + wave] = mine;
                    __syncthreads();
                    const floatx4 f0 = *reinterpret_cast<const floatx4 *>(pt + row * 8), f1 = *reinterpret_cast<const floatx4 *>(pt + row * 8 + 4);
                    wv_w[row] = f(f0, f1);
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int i4 = 0; i4 < 4; ++i4) {
                        const floatx4 x = *reinterpret_cast<const floatx4 *>(wv_w + nb * 32 + 8 * i4 + 4 * g_s);
#pragma unroll
                        for (int j = 0; j < 4; ++j) v[4 * i4 + j] = x[j];
                    }
                };
                auto exponent = [&](float s, float most) {  // (the maximum is subtracted before the scale)
                    float e = fast_exp2((s - most) * a.c);
                    FCS_OPAQUE_V(e);  // (else it is branched around, register by register)
                    return e;
                };
                float most[16], v[16];  // of this lane's keys so far: maximum, and sum relative to it
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    most[i] = kNegBig;
                    v[i] = 0.f;
                }
                sweep(nb, qs, [&](int, const floatx16 &c, auto counts) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const float m = fmaxf(most[i], counts(i) ? c[i] : kNegBig), e = exponent(c[i], m);
                        v[i] = fmaf(v[i], exponent(most[i], m), counts(i) ? e : 0.f);
                        most[i] = m;
                    }
                });
                float rmax[16];
                {
                    float m[16];
#pragma unroll
                    for (int i = 0; i < 16; ++i) m[i] = most[i];
                    reduce(fold_lanes_max(m, lane_s), rmax, [](floatx4 x, floatx4 y) {
                        return fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(y[0], y[1]), fmaxf(y[2], y[3])));
                    });
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) v[i] *= exponent(most[i], rmax[i]);
                reduce(fold_lanes_sum(v, lane_s), v, [&](floatx4 x, floatx4 y) {
                    const float L = ((x[0] + x[1]) + (x[2] + x[3])) + ((y[0] + y[1]) + (y[2] + y[3]));
                    return (row0 + row < a.q_rows) ? __builtin_amdgcn_rcpf(L) : 0.f;
                });
                sweep(nb, qs, [&](int t, const floatx16 &c, auto counts) {
                    float sum = 0.f;
#pragma unroll
                    for (int i = 0; i < 16; ++i) {  // (a row's weight may be NaN: then it must not reach the keys that the row does not see)
                        const float with = fmaf(exponent(c[i], rmax[i]), v[i], sum);
                        sum = counts(i) ? with : sum;
                    }
#pragma unroll
                    for (int u = 0; u < TPW; ++u)  // col_acc lives in registers: static index only
                        if (u == t) col_acc[u] += sum;
                });
            }
            __syncthreads();  // the query rows are read no more: their tile may be rewritten
            FCS_WAIT_VM(0);
            if (gone) {
                const int rot_n = KEEP_ALL || next_key_head ? 0 : rot ^ 1;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const int j = rot_n ? STEPS - 1 - s : s;
                    fetch_item(k_nxt, j / DC, j % DC, j % NS);
                }
            }
        }
        if (!KEEP_ALL) rot = __builtin_amdgcn_readfirstlane(next_key_head ? 0 : (rot ^ 1));
        k_cur = k_nxt;
        cur_rb = nxt_rb;
        cur_hr = nxt_hr;
    }
    FCS_WAIT_VM(0);  // drain the look-ahead fetches before the block's LDS is released

    // ---------------- the two half-waves hold different rows of the same keys: add, then store
    float *dst = a.partial + ((int64_t)(hgi * a.f_nwgq + qwg) * a.B + b) * a.Sk;
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const float v = col_acc[t] + __shfl_xor(col_acc[t], 32);
        if (g == 0 && t <= tmax_lane) dst[tile_first(t) + n] = v;
    }
}

template <int DC, int NB, int TPW, bool NARROW, bool CAUSAL>
static void launch_one(const Plan &p, const Args &a, hipStream_t st)
{
    const dim3 grid(p.f_nwgq * p.B, p.f_hg);
    if (p.bf16) hipLaunchKernelGGL((fcs_tall_kernel<DC, NB, TPW, true, NARROW, CAUSAL>), grid, dim3(512), 0, st, a);
    else hipLaunchKernelGGL((fcs_tall_kernel<DC, NB, TPW, false, NARROW, CAUSAL>), grid, dim3(512), 0, st, a);
}
template <int DC, int NB, int TPW>
static void launch_tpw(const Plan &p, const Args &a, hipStream_t st)
{
    const bool narrow = p.D != DC * 64;
    if (p.causal) narrow ? launch_one<DC, NB, TPW, true, true>(p, a, st) : launch_one<DC, NB, TPW, false, true>(p, a, st);
    else if constexpr (DC == 2 || (NB == 2 && TPW == 4))
        narrow ? launch_one<DC, NB, TPW, true, false>(p, a, st) : launch_one<DC, NB, TPW, false, false>(p, a, st);
}
template <int DC>
static bool launch_dc(const Plan &p, const Args &a, hipStream_t st)
{
    switch (p.f_tpw) {
    case 2: launch_tpw<DC, 2, 2>(p, a, st); break;
    case 3: launch_tpw<DC, 2, 3>(p, a, st); break;
    case 4: launch_tpw<DC, 2, 4>(p, a, st); break;
    case 5: launch_tpw<DC, 1, 5>(p, a, st); break;
    case 6: launch_tpw<DC, 1, 6>(p, a, st); break;
    case 7: launch_tpw<DC, 1, 7>(p, a, st); break;
    case 8: launch_tpw<DC, 1, 8>(p, a, st); break;
    default: return false;
    }
    return true;
}

hipError_t launch_tall(const Plan &p, const Args &a, hipStream_t st)
{
    if (p.Sk < 32 || p.f_kg != 8 || p.f_tpw * 256 < p.Sk || (!p.causal && p.D <= 64 && p.f_tpw != 4)) return hipErrorInvalidValue;
    if (!(p.D > 64 ? launch_dc<2>(p, a, st) : launch_dc<1>(p, a, st))) return hipErrorInvalidValue;
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    return launch_finalize(a, st);
}

size_t describe_tall(const Plan &p, const Args &a, char *buf, size_t n)
{
    const char *bf = p.bf16 ? "true" : "false", *narrow = p.D % 64 ? "true" : "false", *causal = p.causal ? "true" : "false";
    const int r = snprintf(buf, n, "fcs_tall_kernel<%d,%d,%d,%s,%s,%s> grid %d x %d, %d x %d units per workgroup, %d slabs", p.Dp / 64, p.f_tpw > 4 ? 1 : 2, p.f_tpw, bf,
                           narrow, causal, p.f_nwgq * p.B, p.f_hg, p.f_hpg, p.f_rbpw, p.n_partials);
    if (r < 0) return 0;
    const size_t len = (size_t)r;
    return len + describe_finalize(a, false, len < n ? buf + len : nullptr, len < n ? n - len : 0);
}

}  // namespace fcs
