// Launch plan for the column-mean kernels: how one call is cut into workgroups and how
// the caller's workspace is laid out.  Pure host arithmetic, shared by
// fcs_workspace_bytes() and the launch functions so both always agree.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace fcs {

constexpr int kWavesPerBlock = 4;   // 256 threads
constexpr int kStageKeys = 64;      // keys staged in LDS per step of either pass
constexpr int kComputeUnits = 256;  // MI355X
constexpr int kFusedMaxKeys = 2048; // 8 waves x 8 tiles x 32 keys of fp32 scores per 32 query rows
constexpr float kPrescaledMaxScale = 0.1251f;  // single-pass kernels: the operand is pre-scaled up to this |scale| (fp16)
constexpr int kFusedMaxKeys64 = 2560; // 64-wide heads: ten tiles per wave
constexpr int kFusedMaxKeysNarrow = 1536; // heads of 72 .. 120 channels: in every layout and whatever the number of key heads
constexpr int kFewRowsMaxRows = 4;      // few-rows path: at most this many averaged query rows per head ...
constexpr int kFewRowsMaxScores = 12288; // ... and rows * Sk scores (48 KB of LDS)
constexpr int kSmallMaxTiles = 9;        // short-sequence path: one wave holds the scores of 32 rows x (32 x 9) keys
// ... whose workgroups keep the keys of this many heads in an LDS ring (112 KB at most)
constexpr int small_ring_heads(int tiles) { return 28 / tiles < 16 ? 28 / tiles : 16; }

// column pass (fcs_stream_kernels.h): ring slots of 64-key stages and keys per workgroup chunk, sized so
// that the LDS ring plus one accumulator slice per wave fit (twice per compute unit for 4-wave blocks)
constexpr int col_ring_slots(int D, int waves) { return (D == 256 || (D == 128 && waves == 4)) ? 3 : 4; }
constexpr int col_chunk_max(int D, int waves) { return (D == 256) ? 1024 : (D == 128 && waves == 4) ? 1536 : 2048; }

// The shares of a pass (64-key stages): the shortest, and what starting on a row block or unit costs
constexpr int kMinShare = 4;
constexpr int start_places(int D, int rows_per_wave) { return D == 256 ? 1 : (D == 64 && rows_per_wave == 32) ? 3 : 2; }

// row-statistics pass on the same stream (fcs_stream_kernels.h): ring slots
constexpr int row_ring_slots(int D, int waves) { return (D == 256 || waves > 8) ? 3 : 4; }

#if defined(__HIPCC__)
#define FCS_HD __host__ __device__ inline
#else
#define FCS_HD inline
#endif

// Division of 0 <= n < 2^32 by a number that the host knows: a multiply-high and one correction (the estimate is the
// quotient or one less).
struct FastDiv {
    uint32_t d, magic;
    void set(int64_t by)
    {
        d = (uint32_t)by;
        magic = by <= 1 ? 0xffffffffu : (uint32_t)((1ull << 32) / d);
    }
    FCS_HD int quot(int n, int &rest) const
    {
        int q = (int)(((uint64_t)(uint32_t)n * magic) >> 32);
        rest = n - q * (int)d;
        if ((uint32_t)rest >= d) {
            rest -= (int)d;
            ++q;
        }
        return q;
    }
    FCS_HD int quot(int n) const
    {
        int rest;
        return quot(n, rest);
    }
};

// The two-pass path lays the work of a pass out as a line of 64-key stages, head after head and row block after row
// block, and gives every workgroup an equal share of it.  Row block rb of any head has
//     n(rb) = min(last, first + (rb + 1) * step)    stages:
// the stages up to the last key that one of its rows sees.  step is 0 where all row blocks count the same (the line may
// then be counted in units of several stages), else a power of two.  Every row block takes `start` places of the line in front
// of its stages, for what starting on it costs a workgroup.  A line has fewer than 2^31 places.
struct StageLine {
    int first, step, last, log_step, start;
    FCS_HD int n(int rb) const
    {
        const int v = first + (rb + 1) * step;
        return v < last ? v : last;
    }
    // how many of the row blocks before rb have `cap` stages at most
    FCS_HD int up_to(int rb, int cap) const
    {
        if (cap >= last) return rb;
        const int m = (step == 0 || cap < first) ? 0 : (cap - first) >> log_step;
        return m < rb ? m : rb;
    }
    // stages of the row blocks before rb that are among the first `cap` of their block
    FCS_HD int sum(int rb, int cap) const
    {
        const int c = cap < last ? cap : last;
        if (step == 0) return rb * c;
        int m = c > first ? (c - first) >> log_step : 0;  // row blocks that end at or below the cap
        if (m > rb) m = rb;
        return m * first + step * (m * (m + 1) / 2) + (rb - m) * c;
    }
    // places of the row blocks before rb
    FCS_HD int places(int rb) const { return sum(rb, last) + rb * start; }
    // stages lo .. hi-1 of row block rb
    FCS_HD int between(int rb, int lo, int hi) const
    {
        int v = n(rb);
        v = (v < hi ? v : hi) - lo;
        return v > 0 ? v : 0;
    }
    // column pass, chunks of cs stages of a head with nrb row blocks: the row blocks that see chunk c
    FCS_HD int sees(int nrb, int cs, int c) const { return nrb - up_to(nrb, c * cs); }
    // how many chunks every row block sees
    FCS_HD int every(int cs) const { return (n(0) + cs - 1) / cs; }
    // (row block, chunk) pairs among the first `chunks` chunks, of which `all` = every(cs) go without looking
    FCS_HD int pairs(int nrb, int cs, int chunks, int all) const
    {
        int seen = nrb * (chunks < all ? chunks : all);
        for (int c = all; c < chunks && c * cs < last; ++c) seen += sees(nrb, cs, c);
        return seen;
    }
    // places of the first `chunks` chunks; each row block takes `start` places in each chunk that it sees
    FCS_HD int chunk_places(int nrb, int cs, int chunks) const { return sum(nrb, chunks * cs) + pairs(nrb, cs, chunks, every(cs)) * start; }
};

struct Plan {
    int B, H, Sq, Sk, D;
    int Dp;      // head dim the kernels are compiled for: 64, 128 or 256, the smallest that holds D
    int bf16;    // operands are bf16 instead of fp16 (set by the caller after make_plan)
    int q_rows;  // query rows that are averaged: min(cls_n, Sq) or Sq
    int causal, k_past;
    // two-pass path: query heads of a key head whose rows are laid end to end (1: none), and the heads and rows per
    // head that come of it; everything below up to the single-kernel paths counts in those
    int fold, v_heads, v_rows;
    // pass 1: row statistics.  Workgroup w takes the stages [w * r_seg, (w + 1) * r_seg) of the line
    // (batch entry, head, row block)
    int qw;          // query rows per wave (32 or 64)
    int k1_waves;    // waves per block (4 or 8); a block covers k1_waves*qw rows
    int n_qblk;      // row blocks per head
    int rows_pad;    // n_qblk * k1_waves * qw
    StageLine r_line;
    int r_unit, r_seg, r_len, r_blocks;  // stages per unit of the line, units per share and in all, workgroups
    int r_whole;     // every row block lies within one share
    int r_one;       // every share is one (part of a) row block
    FastDiv r_by_seg, r_by_head, r_by_block, by_heads;  // divisions by r_seg, a head's units, a row block's (step 0), v_heads
    // column pass: the same over (batch entry, key chunk, head, row block); a (head, row block) is a unit of the chunk, whose
    // column sums a block keeps in LDS
    int c_nb, c_waves; // 32-row fragments per wave, waves per block: a unit has 32 * c_nb * c_waves rows
    int c_nrb;         // row blocks per head
    int c_chunk, c_nchunks;
    StageLine c_line;
    int c_unit, c_cs;                      // stages per unit of the line, units per chunk
    int c_seg, c_len, c_blocks, c_direct;  // c_direct: block w computes all of chunk w and writes the means
    int c_one;                             // every share is one chunk of one unit
    int c_every;                           // chunks that every row block sees
    FastDiv c_by_seg, c_by_batch, c_by_chunk, c_by_blocks;  // divisions by c_seg, a batch entry's units, c_chunk, c_nrb
    FastDiv c_by_chunks;  // by c_nchunks (c_direct), the chunks that some row sees (c_unit > 1 or c_one), or the places of a
                          // chunk that all row blocks see to its end
    // fused single-kernel path: non-causal, all keys of a row block fit in one
    // workgroup's registers.  grid = (f_nwgq * B, f_hg)
    int fewrows;     // 1: few-rows path (non-causal, q_rows <= 4): grid = B * f_hg, slabs = f_hg
    int small;       // 1: short-sequence path (non-causal, Sk <= 288, D <= 64): grid = B * f_hg, slabs = f_hg,
                     //    f_tpw key tiles, f_nqblk row tiles of 32 rows per head
    int fused;       // 1: use it (then the two-pass fields above are unused)
    int tall;        // with fused: 1: shared query rows (fcs_tall.hip), 64 of them per wave up to four key tiles per wave, 32 beyond
    int f_kg, f_qg;  // waves along keys / along queries, f_kg * f_qg == 8
    int f_tpw;       // 32-key tiles per wave
    int f_nqblk;     // query blocks of 32 * f_qg rows
    int f_hg, f_hpg; // head groups, heads per group
    int f_rbpw;      // adjacent query blocks per workgroup (fused path; 1 on the few-rows path)
    int f_nwgq;      // workgroups along the query axis: ceil(f_nqblk / f_rbpw)
    int n_partials;  // slabs summed by the finalize kernel (two-pass path: at most)
    int gen_blocks;  // two-pass path: resident workgroups of one generation (what the GPU holds at once)
    // workspace layout (byte offsets, each 256-byte aligned)
    size_t off_lse;      // float2 [B*v_heads][rows_pad]  r_whole: row maximum and log2 of the row sum; else the first
                         //                               B*v_heads*n_qblk of the sets of row statistics (row maximum and row sum)
    size_t off_ml;       // float2 [shares][rows of a block]  the rest of them: set w + i is share w's of row block i
    size_t off_partial;  // float  [c_chunk] slabs: w + i is share w's of chunk i (none with c_direct)
    size_t total;
};

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
inline size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Returns false for invalid dimensions.  cls_n <= 0 means all rows.  raw: the single-pass kernels may not take a pre-scaled operand.  Hk: key heads, a divisor of H.
// tight_stages > 0: the two-pass path with as little workspace as it can do with: row blocks are not cut, chunks are not longer
// than that; < 0: not even slabs, a workgroup computes all of a chunk (see plan_within).  few_slabs: in one pass, and 64 rows per wave, also
// where something else is quicker.
inline bool make_plan(Plan &p, int causal, int B, int H, int Hk, int Sq, int Sk, int D, int cls_n, int k_past, int tight_stages = 0,
                      int raw = 0, bool few_slabs = false)
{
    if (B < 1 || H < 1 || Hk < 1 || H % Hk != 0 || Sq < 1 || Sk < 1 || D < 1 || k_past < 0) return false;
    p.B = B; p.H = H; p.Sq = Sq; p.Sk = Sk; p.D = D;
    p.Dp = (D <= 64) ? 64 : (D <= 128) ? 128 : 256;
    p.bf16 = 0;
    p.causal = causal ? 1 : 0;
    p.k_past = causal ? k_past : 0;
    p.q_rows = (cls_n > 0 && cls_n < Sq) ? cls_n : Sq;

    // ---- grouped key heads: the rows of all query heads of a key head can be laid end to end, as one head whose keys
    // are then streamed once per row block of that head instead of once per query head (and row block).  For at most 128
    // averaged rows, the smallest row block: more of them fill their own blocks, and a causal block that holds rows
    // of several heads cannot stop at its own last key (Q 200, 32 on 4 heads, K 6000, D 64: 48 us head by head, 49
    // folded).  Below that it pays
    //  * where the rows of a batch entry then form a single unit of the column pass: no slabs, no final reduction
    //    (16 on 1 head, Q 8, K 1000, D 64: 15.4 us folded, 17.8 head by head), and
    //  * from a number of workgroups on that the call has head by head at the finest key split (visible keys / 256): one
    //    per compute unit while half of a block's rows or more are missing (measured nearly equal or slower up to 256,
    //    5 .. 20 % faster from 288 on, whatever the head dim), more when less is saved: ten for blocks with 65 .. 128 rows
    //    of 128 (D 64 and 128: 0.84 .. 0.97 of the speed at 1500, 1.0 at 2500 .. 3000, 1.01 .. 1.18 at 4096), two for
    //    256-wide heads, whose row pass has blocks of 128 rows either way (0.94 .. 1.0 at 320 .. 384, 1.0 .. 1.26 at 512).
    // B 4, 32 on 8 heads, K 8192, D 128 bf16: Q 64 94.7 us head by head, 54.2 folded, Q 128 1.16 times as fast.
    const int G = H / Hk;
    const int seen_keys = p.causal ? (int)((long)p.k_past + p.q_rows < Sk ? (long)p.k_past + p.q_rows : Sk) : Sk;
    const long head_blocks = (long)B * H * ceil_div(seen_keys, 4 * kStageKeys);
    const long worth = (p.q_rows <= 64) ? kComputeUnits + 1 : (p.Dp == 256 ? 2 : 10) * kComputeUnits;
    const bool one_unit = Hk == 1 && (long)G * p.q_rows <= 128;
    p.fold = (G > 1 && p.q_rows <= 128 && (long)G * p.q_rows * p.q_rows < (1L << 31) && (one_unit || head_blocks >= worth)) ? G : 1;
    p.v_heads = H / p.fold;
    p.v_rows = p.q_rows * p.fold;

    // ---- rows per block of both passes: 512 (8 waves x 64 rows), 256 or 128 (4 waves x 64 or 32).
    // Taller blocks re-read the keys less often.  A small call takes a shorter block instead, while
    // even the finest key split (256 keys per block) of the taller one would leave most compute units
    // without a block: B 1, H 16, S 512, D 128 ran as 32 blocks of 512 rows, 13.6 + 16.0 us.
    int block_rows = (p.v_rows > 256) ? 512 : (p.v_rows > 128) ? 256 : 128;
    while (block_rows > 128 &&
           (long)ceil_div(p.v_rows, block_rows) * B * p.v_heads * ceil_div(Sk, 4 * kStageKeys) < kComputeUnits)
        block_rows /= 2;

    // ---- pass 1
    p.qw = (block_rows > 128) ? 64 : 32;
    p.k1_waves = (block_rows > 256) ? 8 : 4;
    if (p.Dp == 256) { p.qw = 32; p.k1_waves = 4; }  // the stationary rows of a wider head fill the registers sooner
    const int qblk = p.k1_waves * p.qw;
    p.n_qblk = ceil_div(p.v_rows, qblk);
    p.rows_pad = p.n_qblk * qblk;
    // ---- the stages of a pass.  A causal row block ends at the last key that one of its rows sees; of a call with a
    // single row block per head (or rows laid end to end: every block holds a head's last row) that is the same for all.
    const auto line_of = [&](int rows, int blocks, int past) {
        const int seen = p.causal ? (int)((long)past + p.q_rows < Sk ? (long)past + p.q_rows : Sk) : Sk, n = ceil_div(seen, kStageKeys);
        if (!p.causal || p.fold > 1 || blocks == 1) return StageLine{n, 0, n, 0, 0};
        const int step = rows / kStageKeys;  // 2, 4 or 8
        return StageLine{ceil_div(past < Sk ? past : Sk, kStageKeys), step, n, step == 8 ? 3 : step == 4 ? 2 : 1, 0};
    };
    // One generation of workgroups: an 8-wave block fills a compute unit's registers, the 4-wave blocks fit twice
    // (256-wide heads: the kernels' registers and LDS allow one block per compute unit whatever its waves).
    p.gen_blocks = (p.k1_waves == 8 || p.Dp == 256) ? kComputeUnits : 2 * kComputeUnits;

    // A line of 2^31 places (20 s of a pass on 512 rows of 128 channels) or more has no shares: a workgroup per row block in pass 1
    // (or, where all are equal, whole ones), and per chunk in the column pass.  The limit leaves room for rounding up to whole shares.
    const auto stages_of = [&](const StageLine &l, int blocks) {
        double t = 0.;
        for (int rb = 0; l.step && rb < blocks; ++rb) t += l.n(rb);
        return (l.step ? t : (double)l.last * blocks) * B * p.v_heads;
    };
    constexpr double kMostPlaces = 2.1e9;

    // ---- pass 1: equal shares of the line, at least kMinShare stages each.  A share that crosses into another row block
    // pays that block's start (Q fragments, first key stages) on top, so where all row blocks are equal it is also
    // priced to cut each of them into equal parts, or to give a workgroup whole ones.
    {
        const long blocks = (long)p.n_qblk * B * p.v_heads;
        if (blocks >= (1L << 31)) return false;
        const int start = start_places(p.Dp, p.qw);
        p.r_line = line_of(qblk, p.n_qblk, p.k_past);
        p.r_unit = 1;
        const double all = stages_of(p.r_line, p.n_qblk) + (double)blocks * start;
        const bool huge = all >= kMostPlaces || tight_stages != 0;
        int seg = huge ? 0 : (int)(((int64_t)all + p.gen_blocks - 1) / p.gen_blocks);
        if (seg < kMinShare + start) seg = kMinShare + start;
        p.r_whole = p.r_one = 0;
        p.r_line.start = start;
        const int best = seg + start;  // (a share that starts inside a row block pays its start unasked)
        {
            const int n = p.r_line.last;
            // whole row blocks per workgroup (uneven ones without shares: one, and the hardware hands them out)
            const long per = (huge && p.r_line.step) ? 1 : (blocks + p.gen_blocks - 1) / p.gen_blocks;
            const int most = ceil_div(n, kMinShare);
            const long fit = p.gen_blocks / blocks;
            const int parts = (per > 1 || fit < 2 || tight_stages != 0) ? 1 : (int)(fit < most ? fit : most);
            const int part = ceil_div(n, parts);
            // (row blocks that see different numbers of keys: parts of the longest one's length)
            if (huge || ((p.r_line.step == 0 || per == 1) && per * (part + start) <= best)) {
                seg = (int)per;
                p.r_unit = part;
                const int units = ceil_div(n, part);
                p.r_whole = units == 1;
                p.r_one = per == 1;
                p.r_line = StageLine{units, 0, units, 0, 0};
            }
        }
        p.r_len = B * p.v_heads * p.r_line.places(p.n_qblk);
        if (seg > p.r_len) seg = p.r_len;
        p.r_seg = seg;
        p.r_blocks = ceil_div(p.r_len, seg);
        p.r_by_seg.set(seg);
        p.r_by_head.set(p.r_line.places(p.n_qblk));
        p.r_by_block.set(p.r_line.last + p.r_line.start);
        p.by_heads.set(p.v_heads);
    }

    // ---- column pass (streaming kernel)
    int64_t slab_stages = 0;  // what the call's slabs take of the workspace, in stages of 64 floats
    {
        if (block_rows > 256) { p.c_nb = 2; p.c_waves = 8; }
        else if (block_rows > 128) { p.c_nb = 2; p.c_waves = 4; }
        else { p.c_nb = 1; p.c_waves = 4; }
        if (p.Dp == 256) { p.c_nb = 1; p.c_waves = (block_rows > 128) ? 8 : 4; }
        const int rows = 32 * p.c_nb * p.c_waves;
        p.c_nrb = ceil_div(p.v_rows, rows);
        const int start = start_places(p.Dp, 32 * p.c_nb);
        const long units = (long)p.v_heads * p.c_nrb;  // per batch entry
        int most = col_chunk_max(p.Dp, p.c_waves) / kStageKeys;
        if (tight_stages > 0 && tight_stages < most) most = tight_stages;
        const long target = (p.c_waves == 8 || p.Dp == 256) ? kComputeUnits : 2 * kComputeUnits;
        enum { kShares, kUnits, kDirect };
        struct Split { int cs, seg, how; int64_t slabs; };
        // the cheapest split of a line among those whose slabs take `room` stages at most
        const auto cheapest = [&](const StageLine &stages, int64_t room) {
            const int n = stages.last;
            const double all = stages_of(stages, p.c_nrb);
            // what the final reduction takes, in stages: a launch, and the slabs (one per workgroup and chunk that it touches), written
            // and read.  (With the workgroups alone, calls of many batch entries got a slab per chunk where a workgroup per chunk is as
            // fast without: B 594, H 2, S 189291, 1 row 436 MiB of them.)
            const auto reduce = [&](long slabs, int c) { return 2.5 + (double)slabs * c * 1e-4; };
            // Causal row blocks that see almost the same keys (the last rows of a long context) are quicker whole, four of one head
            // re-reading its chunk, than in shares that straddle two heads at every workgroup (us per call, shares -> whole: H 8, Q 4096,
            // K 65536, D 64 693 -> 653; H 32, Q 1500, K 32768, D 64 538 -> 496; H 4, Q 2048, K 65536, D 128 291 -> 279), up to
            // about 3 % of the line's length (H 12, Q 4096, K 12288, D 128, where whole ones are 14 % longer: 280 in shares, 301).
            const double uneven = stages.step ? 1.03 : 1.;
            const int parts0 = ceil_div(n, most), parts_end = ceil_div(n, kMinShare);
            Split s{1, 1, kDirect, 0};
            double best = 1e300;
            for (int parts = parts0; parts <= parts_end && parts < parts0 + 128; ++parts) {
                const int c = ceil_div(n, parts);
                if (ceil_div(n, c) != parts) continue;
                const long pieces = (long)B * parts * units;  // chunks of the units
                const bool huge = all + (double)pieces * start >= kMostPlaces || tight_stages < 0;
                const auto slabs = [&](long shares) { return (shares + (int64_t)B * ceil_div(Sk, c * kStageKeys)) * c; };
                if (!huge) {
                    StageLine l = stages;
                    l.start = start;
                    const int64_t len = (int64_t)B * p.v_heads * l.chunk_places(p.c_nrb, c, parts);
                    int sg = (int)((len + target - 1) / target);
                    if (sg < kMinShare + start) sg = kMinShare + start;
                    const int64_t need = slabs((len + sg - 1) / sg);
                    const double cost = uneven * (sg + start) + reduce(target + (long)B * parts, c);
                    if (cost < best && need <= room) { best = cost; s = Split{c, sg, kShares, need}; }
                }
                // whole ones per workgroup, priced as if all were as long as the longest
                const long per = (pieces + target - 1) / target;
                if (!huge) {
                    const int64_t need = slabs((pieces + per - 1) / per);
                    const double cost = (double)per * (c + start) + reduce(pieces / per + (units % per ? (long)B * parts : 0), c);
                    if (cost < best && need <= room) { best = cost; s = Split{c, (int)per, kUnits, need}; }
                }
                // a workgroup per chunk, which writes the means itself: no slabs, no final reduction
                const double cost = (double)((B * (long)parts + target - 1) / target) * (double)units * (c + start);
                if (cost <= best) { best = cost; s = Split{c, 1, kDirect, 0}; }
                if (pieces > 4 * target && parts > parts0 + 8) break;
            }
            return s;
        };
        const StageLine stages = line_of(rows, p.c_nrb, p.k_past);
        Split split;
        if (!p.causal) {
            split = cheapest(stages, INT64_MAX);
            slab_stages = split.slabs;
        } else {
            // The workspace's size must not depend on k_past (fcs_workspace_bytes does not know it).  There is room for what the call takes
            // with the usual k_past and with every key visible, and for slabs of up to 8 MiB if one for each chunk fits in there; with
            // another k_past it is split so that it fits.
            const auto same = [](const StageLine &a, const StageLine &b) { return a.first == b.first && a.step == b.step && a.last == b.last; };
            const StageLine usual = line_of(rows, p.c_nrb, Sk > Sq ? Sk - Sq : 0), whole = line_of(rows, p.c_nrb, Sk);
            const Split of_usual = cheapest(usual, INT64_MAX), of_whole = same(usual, whole) ? of_usual : cheapest(whole, INT64_MAX);
            const int64_t all_stages = ceil_div(Sk, kStageKeys), c_most = all_stages < most ? all_stages : most;
            const int64_t shares = B * units * ceil_div((int)all_stages, kMinShare);
            slab_stages = (target < shares ? target : shares) * c_most + B * (all_stages + c_most);  // the most that any k_past takes
            const int64_t small = (8 << 20) / (int64_t)(sizeof(float) * kStageKeys);
            if (slab_stages > small) slab_stages = B * all_stages <= small ? small : 0;
            if (slab_stages < of_usual.slabs) slab_stages = of_usual.slabs;
            if (slab_stages < of_whole.slabs) slab_stages = of_whole.slabs;
            split = same(stages, usual) ? of_usual : same(stages, whole) ? of_whole : cheapest(stages, slab_stages);
        }
        const int n = stages.last, cs = split.cs, how = split.how;
        int seg = split.seg;
        const int used = ceil_div(n, cs);  // chunks that some row sees
        p.c_chunk = cs * kStageKeys;
        p.c_nchunks = ceil_div(Sk, p.c_chunk);
        p.c_line = stages;
        p.c_line.start = start;
        p.c_unit = 1;
        p.c_cs = cs;
        if (how != kShares) {  // counted in chunks (the kernel stops a unit at the last key that it sees)
            p.c_line = StageLine{used, 0, used, 0, 0};
            p.c_unit = cs;
            p.c_cs = 1;
        }
        const long chunks = (long)B * p.c_nchunks;
        if (chunks >= (1L << 31)) return false;
        p.c_direct = how == kDirect;
        p.c_one = how == kUnits && seg == 1;
        p.c_by_blocks.set(p.c_nrb);
        p.c_len = p.c_seg = p.n_partials = 1;
        p.c_blocks = (int)chunks;
        p.c_by_batch.set(1);
        if (how != kDirect) {
            const int per_batch = p.v_heads * p.c_line.chunk_places(p.c_nrb, p.c_cs, used);
            p.c_len = B * per_batch;
            if (seg > p.c_len) seg = p.c_len;
            p.c_seg = seg;
            p.c_blocks = ceil_div(p.c_len, seg);
            p.n_partials = p.v_heads * p.c_line.chunk_places(p.c_nrb, p.c_cs, 1) / seg + 2;  // of the first chunk, the most seen
            p.c_by_batch.set(per_batch);
        }
        p.c_by_seg.set(p.c_seg);
        p.c_every = p.c_line.every(p.c_cs);
        p.c_by_chunks.set(p.c_direct ? p.c_nchunks : (p.c_unit > 1 || p.c_one) ? used : (int64_t)units * (p.c_cs + p.c_line.start));
        p.c_by_chunk.set(p.c_chunk);
    }

    // ---- few-rows path: a batch of matrix-vector products, one workgroup per (batch entry, head group)
    p.fewrows = 0;
    p.small = 0;
    p.fused = 0;
    p.tall = 0;
    // (One workgroup streams a whole key head and computes its R x Sk scores on the VALU.  The fused
    // path, which splits a head's keys over eight waves and uses the matrix pipe, is quicker when
    // there are fewer (batch entry, head) pairs than compute units and a thousand keys or more per
    // head (B 8, H 16, S 2048, 4 rows: 24 -> 15 us), and when a head has more than 4096 scores
    // (B 16, H 16, S 2048, 4 rows: 24.4 -> 19.9 us).  The CLS-token shape B 32, H 16, S 577, 1 row
    // stays here: 13.4 us of kernels against 15.8 us on the fused path.)
    const bool fused_is_quicker = D == 64 && Sk <= kFusedMaxKeys &&
                                  ((Sk >= 1024 && (long)B * H < kComputeUnits) || (long)p.q_rows * Sk > 4096);
    if (!causal && p.q_rows <= kFewRowsMaxRows && (long)p.q_rows * Sk <= kFewRowsMaxScores && (D == 64 || D == 128) &&
        !fused_is_quicker) {
        p.fewrows = 1;
        p.fold = 1;
        const long bh = (long)B * H;
        int hpb = (int)((bh + 2047) / 2048);  // heads per workgroup: about 2048 workgroups at most
        if (hpb > H) hpb = H;
        p.f_hpg = hpb;
        p.f_hg = ceil_div(H, hpb);
        p.f_rbpw = 1;
        p.f_nwgq = 1;
        p.n_partials = p.f_hg;
        p.off_lse = p.off_ml = p.off_partial = 0;
        p.total = align256(sizeof(float) * (size_t)p.n_partials * B * Sk);
        return (long)B * p.f_hg < (1L << 31);
    }

    // ---- short-sequence path: a wave holds all the keys of its 32 rows, a workgroup owns f_hpg heads of a
    // batch entry and deals their (head, 32-row tile) items to its eight waves, eight per step
    if (!causal && Sk <= 32 * kSmallMaxTiles && D <= 64) {
        const int tiles = ceil_div(Sk, 32), rt = ceil_div(p.q_rows, 32);
        // the keys of the heads that two consecutive steps touch must fit the ring: items 8t .. 8t + 15
        int span = 0;
        for (int t = 0; t < rt; ++t) {
            const int c = (8 * t + 15) / rt - (8 * t) / rt + 1;
            if (c > span) span = c;
        }
        if (span <= small_ring_heads(tiles)) {
            p.small = 1;
            p.fold = 1;
            p.f_tpw = tiles;
            p.f_nqblk = rt;
            // Heads per workgroup: one workgroup is resident per compute unit, so the launch runs in generations
            // of kComputeUnits workgroups, each as long as its steps plus about one step for starting and finishing.
            p.f_hpg = H;
            double best = 0.;
            for (int hg = 1, hpg = H; hpg >= 1; hg = (hpg > 1) ? ceil_div(H, hpg - 1) : H + 1, hpg = (hg <= H) ? ceil_div(H, hg) : 0) {
                const long gens = ((long)B * hg + kComputeUnits - 1) / kComputeUnits;
                const double cost = (double)gens * (ceil_div(hpg * rt, 8) + 1.0) + 0.01 * hg;
                if (hg == 1 || cost < best) {
                    best = cost;
                    p.f_hpg = hpg;
                }
            }
            p.f_hg = ceil_div(H, p.f_hpg);
            p.f_rbpw = 1;
            p.f_nwgq = 1;
            p.f_kg = 1;
            p.f_qg = 8;
            p.n_partials = p.f_hg;
            p.off_lse = p.off_ml = p.off_partial = 0;
            p.total = align256(sizeof(float) * (size_t)p.n_partials * B * Sk);
            return (long)B * p.f_hg < (1L << 31);
        }
    }

    // ---- fused path
    // (at least one whole key tile: the kernel moves a tile that reaches past the last key back to end there)
    // (64-wide kernels for head dims up to 64, 128-wide ones up to 128; wider heads take the two-pass path)
    // (Heads of 72 .. 120 channels: us per call beyond 1536 keys, two passes -> one: B 8 H 16 S 2000 D 96 299 -> 219, S 1700 D 80 230 -> 155,
    // D 120 260 -> 201, B 3 H 12 S 1900 D 72 87 -> 60.  Up to 63 tiles: 2017 .. 2048 keys would gain as much, S 2048 D 96 287 against 230, and
    // have not been moved yet.)
    const bool narrow128 = D > 64 && D < 128;
    // (64-wide heads: the shared-Q variants hold ten tiles per wave, so calls of up to 2560 keys are served too, unless grouped
    // heads are laid end to end, whose keys are streamed once for the whole group.  us per call, two passes -> here:
    // B 1 H 16 S 2500 47.9 -> 33.5, B 4 H 16 S 2300 212.8 -> 88.0, H 1 S 2500 14.6 -> 10.9, 5 averaged rows of B 8 H 16
    // S 2300 30.2 -> 12.1, 128 of them 29.9 -> 18.5; no size in between was slower.)
    const bool wide = D == 64 && tight_stages == 0;
    // Heads of 72 .. 120 channels beyond 1536 keys, in two passes:
    //  * with tight_stages.  The single pass has the same slabs in every layout, and the row statistics that two passes can do with are
    //    mostly less: B 32 H 16 S 1537 D 96 10.5 MiB and 8.
    //  * many more (batch entry, head) pairs than compute units, with few rows each.  Each unit then reads a key head of its own, and those
    //    that an XCD reads at a time are many times its L2.  us per call, two passes against one, K 1600, D 120 unless stated: B 32 H 32
    //    Q 64 134 against 92, Q 128 182 against 197, Q 256 271 against 326, Q 512 476 against 529 (D 96 Q 128 0.93 of two passes' time, Q 256
    //    1.09, Q 512 0.99; D 72 Q 256 0.95; half as many pairs Q 256 1.20, Q 512 1.10).
    //    Rows laid end to end read a key head once for all its query heads: 32 on 8 heads B 32 Q 32 52.6 against 50.6, Q 64 76 against
    //    88, Q 128 125 against 162 (D 96 119 against 131, D 72 0.91; 32 on 16 Q 32 0.69, Q 64 1.04, 32 on 4 Q 4 1.57, D 72 1.28; with half as
    //    many pairs Q 4 1.00, Q 128 0.96).  Beyond 128 rows they are not laid so, and one pass is quicker: Q 256 0.84.
    const long pairs = (long)B * H;
    const bool crowded = narrow128 && !few_slabs && pairs > kComputeUnits &&
                         (p.fold > 1 ? pairs > 2 * kComputeUnits && (p.q_rows > 32 ? D > 80 : p.fold > 2)
                                     : Hk == H && p.q_rows >= 128 && p.q_rows <= 512 && D > (p.q_rows % 256 == 0 ? 80 : 96));
    const int fused_max = !narrow128 ? ((wide && p.fold == 1) ? kFusedMaxKeys64 : kFusedMaxKeys)
                          : tight_stages == 0 && !crowded ? 63 * 32 : kFusedMaxKeysNarrow;
    // Causal calls of 257 .. 2048 keys whose heads are not laid end to end: the same, a mask on the tiles that the diagonal crosses and no
    // exponents behind it.  Two passes cost three launches and both products for what is mostly latency; us per call, two passes -> here:
    // up to 1024 keys, 64 rows per wave: H 32 S 1000 D 128 31.7 -> 20.7, H 16 S 800 D 64 21.1 -> 12.0, H 16 Q 100 K 1000 D 128 17.6 -> 12.1,
    // H 2 S 300 D 128 14.8 -> 10.5; beyond, 32 rows: H 32 S 1500 D 128 47.6 -> 38.9, S 1200 D 64 36.2 -> 22.6, Q 128 K 2048 H 64 24.8 -> 17.0,
    // H 64 S 1700 97.5 -> 86.8, H 96 S 1536 101.9 -> 99.8.  With rows out of range: see the rare path of fcs_tall.hip.
    // Long prompts of many heads fill the chip in two passes, which leave out the products behind the diagonal too, two passes against one:
    // D 128, S 2048 H 96 153 against 173, H 64 106 against 111, H 48 86 and 86, H 32 60.2 against 61.4, H 24 54.3 against 48.0; S 1900 H 64
    // 103.5 against 107.8, H 32 60.9 against 59.3; D 64, H 96 106 against 111, H 64 75.9 and 75.6; Q 1024 K 2048 H 64 79.8 against 62.1.
    // (One batch entry, as prompts and windows are.  Batches would gain as much, two passes against one: B 64 H 16 S 1024 D 64 336 against
    // 265, B 16 H 12 S 700 D 80 86 against 47, though not B 4 H 32 S 2048 D 128, 191 against 227; they have not been moved yet.)
    const bool long_prompt = Sk > 1792 && 2L * (Sk - Sq) < Sq && (long)B * H * ceil_div(p.q_rows, 32) >= (D > 64 ? 2000 : 4200);
    const bool causal_single = causal && B == 1 && p.fold == 1 && D <= 128 && Sk > 256 && Sk <= 2048 && !long_prompt;
    if (causal_single || (!causal && Sk >= 32 && Sk <= fused_max && D <= 128)) {
        p.fused = 1;
        p.fold = 1;
        const int tiles = ceil_div(Sk, 32);
        int usual = 1;  // key groups: the fewest that hold the keys with eight tiles per wave
        while (usual * 8 < tiles && usual < 8) usual *= 2;
        if (narrow128) while (usual * 6 < tiles && usual < 8) usual *= 2;  // six there
        // Other splits over the key groups are priced too; tight_stages keeps the usual one, whose slabs are what such a
        // caller has always had room for.
        //  * Half as many groups of nine or ten tiles (64-wide heads): half the barriers, row sums and exchanges, but the last
        //    generation is coarser, and a unit of ten tiles takes 1.9 times one of five, not 1.6 as eight do.  us per call,
        //    usual -> half: B 8 H 16 S 1100 50.2 -> 44.0, B 32 H 16 S 577 57.2 -> 52.8, S 1040 173.6 -> 156.4, but B 32 H 12
        //    S 640 44.4 -> 48.4 and B 1 H 12 S 1100 12.7 -> 14.0: both sides of the price below.
        //  * More groups of fewer tiles where the workgroups get two units at most, i.e. where most of the chip is idle or a
        //    unit's chain of tiles is all there is: B 2 H 4 S 512 9.3 -> 7.3, B 1 H 16 S 1024 bf16 14.1 -> 12.3, D 128
        //    18.2 -> 15.1, B 8 H 8 S 197 D 128 11.3 -> 8.7.  With three units or more it was up to 9 % slower.
        // 64 query rows per wave and eight key groups (fcs_tall.hip), up to 1024 keys.  us per call, 32 rows -> 64:
        //  * heads of 65 .. 128 channels, from 449 keys on (narrower than 128: 385): B 8 H 16 S 1024 D 128 67.2 -> 53.0, D 96 72.1 -> 50.8;
        //    S 768 40.3 -> 33.5, S 640 31.2 -> 29.1; with two tiles per wave S 512 B 32 75.2 -> 65.5, S 480 B 16 37.7 -> 33.2, but
        //    S 448 B 8 20.2 -> 20.8, S 384 B 32 47.3 -> 54.2 (D 128; D 96, S 400 62.1 -> 51.6).
        //  * 64 channels from 897 keys on where type or scale keep the operand from being pre-scaled: bf16 B 64 H 16 S 1024 252 -> 236, B 16 S 900 63.0 -> 60.1,
        //    but S 800 52.5 -> 53.7, S 577 33.1 -> 35.3, S 512 B 32 40.4 -> 46.4, B 21 H 4 S 887 23.1 -> 23.2; fewer channels from 769 on: D 32
        //    B 16 S 1000 68.8 -> 61.1, D 48 B 32 H 12 S 800 81.6 -> 78.7, but D 48 S 500 24.1 -> 25.8.
        //  * 65 .. 128 channels beyond 1024 keys, with 32 rows per wave: B 8 H 16 D 128 S 2048 248 -> 226, S 1370 128 -> 118, B 64 H 8
        //    S 1200 407 -> 376, Q 32 K 2048 18.6 -> 16.8; H 1 S 2048 13.5 -> 12.8; against the narrow variant of the shorter blocks D 120 S 1700
        //    212.9 -> 199.3, but D 72 B 3 H 12 S 1900 62.5 -> 64.7, B 12 H 32 Q 145 K 1433 D 80 62.7 -> 64.7 (64 channels: S 2048 123.9 against 134.9).
        // Up to 1024 keys, one generation of row blocks of 64 has to stand for nearly one and a half of the shorter ones at least, or those fill
        // the chip better: B 2 H 4 S 1024 D 128 10.4 against 11.1, B 8 H 12 Q 147 K 753 (288 blocks, 480 shorter ones) 13.3 against 14.5, but
        // B 12 H 6 Q 255 K 578 (288, 576) 15.0 -> 13.8, B 9 H 24 Q 69 K 598 (432, 648) 16.5 -> 15.1.  (Up to 64 channels the splits over more waves
        // below have calls of two units per workgroup.)  Up to 64 channels what is gained is the keys, fetched once for a workgroup's row
        // blocks: not with one of them (B 31 H 32 Q 50 K 792 D 48 23.1 against 24.7), and below 897 keys not with few
        // (B 40 H 8 Q 153 K 806 D 48 20.6 against 21.9; B 8 H 12 S 785 D 32 0.93 of the shorter blocks' time, B 14 H 8 S 811 D 48 0.97).
        const auto generations = [&](int rows) { return ((long)B * H * ceil_div(p.q_rows, rows) + kComputeUnits - 1) / kComputeUnits; };
        const auto tall_pays = [&]() {
            if (tight_stages != 0 || tiles > 64) return false;
            if (tiles > 32) return D > 64;
            if (p.q_rows <= 32) return false;
            if (D > 64) return tiles > (narrow128 ? 12 : 14) && (few_slabs || 10 * generations(32) >= 14 * generations(64));
            if (few_slabs) return D < 64 && tiles > 24;
            return (D < 64 || raw) && p.q_rows > 64 && generations(64) > 2 && (tiles > 28 || (D < 64 && tiles > 24 && p.q_rows > 384));
        };
        const bool tall = causal_single || tall_pays();
        double best_kg = 0.;
        bool any = false;
        for (int kg = tall ? 8 : (wide && usual >= 4 && usual * 5 >= tiles) ? usual / 2 : usual; kg <= 8; kg *= 2) {
            const int tpw = ceil_div(tiles, kg), nqblk = ceil_div(p.q_rows, tall ? (tiles > 32 ? 32 : 64) : 32 * (8 / kg));
            if (!tall && kg > usual && (tight_stages != 0 || (long)B * H * nqblk > 2 * kComputeUnits)) break;
            // Units per workgroup: a unit is one (query block, head); a workgroup takes f_rbpw adjacent
            // query blocks times f_hpg heads.  One workgroup is resident per compute unit, so the launch
            // runs in generations of kComputeUnits workgroups, each as long as its units plus about 0.7 of
            // a unit for starting and finishing.  Fewer units per workgroup fill the last generation
            // better (528 workgroups of 16 units take three generations, 2112 of 4 take nine quarter-
            // length ones) at the price of more starts and more partial slabs; more units per workgroup
            // save starts (512 workgroups of 16 units take two generations, 256 of 32 one).
            int best_hpg = H, best_rbpw = 1;
            double best = 0.;
            bool first = true;
            for (int rbpw = 1; rbpw <= 16 && (rbpw == 1 || rbpw <= nqblk); ++rbpw) {
                const int nwgq = ceil_div(nqblk, rbpw);
                if (ceil_div(nqblk, nwgq) != rbpw) continue;  // same grouping as a smaller rbpw
                // heads per workgroup, descending, one value per distinct grouping: hpg = ceil(H / hg) for
                // hg = 1, then the next hg that lowers it (about 2 sqrt(H) values)
                for (int hg = 1, hpg = H; hpg >= 1; hg = (hpg > 1) ? ceil_div(H, hpg - 1) : H + 1, hpg = (hg <= H) ? ceil_div(H, hg) : 0) {
                    const long gens = ((long)nwgq * B * hg + kComputeUnits - 1) / kComputeUnits;
                    // a unit that follows another row block of the same head finds half of its key tiles in
                    // the LDS ring (the shared-Q kernels; measured 4 % of a unit): row blocks per head count
                    // a little less than heads
                    double cost = (double)gens * ((double)hpg * (rbpw - 0.04 * (rbpw - 1)) + 0.7) + 0.01 * hg + 0.002 * rbpw;
                    // The 32 workgroups that an XCD runs at a time are neighbours in launch order: nwgq of
                    // them share a batch entry, i.e. one head's keys.  When the key heads they stream at
                    // the same time outgrow the XCD's 4 MiB L2, the re-reads of a head's keys by its row
                    // blocks miss (measured +6 % at B 256, S 1024 with 32 batch entries per XCD).
                    const long streams = (nwgq >= 32) ? 1 : (32 + nwgq - 1) / nwgq;
                    if (streams * (long)Sk * (2 * p.Dp) > (5L << 19)) cost *= 1.08;
                    if (first || cost < best) {
                        first = false;
                        best = cost;
                        best_hpg = hpg;
                        best_rbpw = rbpw;
                    }
                }
            }
            best *= tpw > 8 ? 1.03 * (tpw + 3) : tpw + 2;  // a unit's time: its tiles, and its reduction
            if (!any || best < best_kg) {
                any = true;
                best_kg = best;
                p.f_kg = kg;
                p.f_qg = 8 / kg;
                p.f_tpw = tpw;
                p.f_nqblk = nqblk;
                p.f_hpg = best_hpg;
                p.f_rbpw = best_rbpw;
            }
        }
        p.tall = tall;
        p.f_hg = ceil_div(H, p.f_hpg);
        p.f_nwgq = ceil_div(p.f_nqblk, p.f_rbpw);
        p.n_partials = p.f_hg * p.f_nwgq * p.f_qg;
        p.off_lse = p.off_ml = p.off_partial = 0;
        p.total = align256(sizeof(float) * (size_t)p.n_partials * B * Sk);
        return (long)p.f_nwgq * B * p.f_hg < (1L << 31);
    }

    // ---- workspace.  A causal call's parts of row blocks, too, are given room for the most that any k_past leaves: a workgroup
    // leaves one set of row statistics per row block that it touches (with a block that is cut, one more than the cuts).
    const int64_t r_most = (int64_t)B * p.v_heads * p.n_qblk * ceil_div(ceil_div(Sk, kStageKeys), kMinShare);
    const int64_t row_sets = p.causal ? (r_most < p.gen_blocks ? r_most : p.gen_blocks) : p.r_whole ? 0 : p.r_blocks;
    size_t off = 0;
    p.off_lse = off;
    off = align256(off + 2 * sizeof(float) * (size_t)B * p.v_heads * p.rows_pad);
    p.off_ml = off;
    off = align256(off + 2 * sizeof(float) * (size_t)qblk * (size_t)row_sets);
    p.off_partial = off;
    off = align256(off + sizeof(float) * kStageKeys * (size_t)slab_stages);
    p.total = off;
    return true;
}

// The plan of a non-causal call for a workspace of `bytes`: the usual one, or one that needs less.  False if none fits, i.e. if the
// row statistics alone (or the slabs of a single-kernel path) do not.
inline bool plan_within(Plan &p, size_t bytes, int B, int H, int Hk, int Sq, int Sk, int D, int cls_n)
{
    const int tight[] = {0, 32, 16, 8, 4, 2, 1, -1};
    for (const int stages : tight) {
        if (!make_plan(p, 0, B, H, Hk, Sq, Sk, D, cls_n, 0, stages)) return false;
        if (p.total <= bytes) return true;
    }
    // (slabs may fit where row statistics do not: B 487 H 19 S 1884 D 104, 153 averaged rows, 3.5 MiB and 18; B 159 H 16
    // S 868 D 8, 126 of them, 4.2 and 8.4 with the shorter blocks)
    return make_plan(p, 0, B, H, Hk, Sq, Sk, D, cls_n, 0, 0, 0, true) && p.total <= bytes;
}

}  // namespace fcs
