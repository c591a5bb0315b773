// Top-k / threshold selection over the fp32 column means, on the GPU and on the caller's stream.
//
// The consumer of the column means is token-importance ranking for pruning (reference:
// README.md:10): it wants the k most-attended key positions of every batch row.  Selecting on the
// kernels' fp32 means, right behind the final reduction and without a host round trip, keeps the
// small means of long contexts that the reference's fp16 result flushes to zero
// (reference: flash_colsum/kernel_causal.py:124).
//
// One workgroup of 1024 threads per batch row.  Wave w owns the w-th sixteenth of the row, E elements per
// lane, and keeps them in registers (rows of up to 32768 entries; longer ones are re-read from the L2 for
// every sweep).  A call is a chain of sweeps over so little data that barriers and LDS round trips are what
// it costs, so the sweeps are few and none has a barrier inside:
//   1. smallest and largest key of the row.  Floats are ordered through the usual monotone map to unsigned
//      integers.
//   2. selection of the k-th largest key: 2048-bin histograms (LDS atomics on integers).  The first one spans
//      exactly [smallest, largest], so that the entries of a row, which share their leading bits, spread over the
//      bins instead of meeting in a few of them (a wave's atomics on one address are served one after the
//      other); each further one spans the bin that holds the k-th key.  It ends when that bin is taken whole:
//      two sweeps for a typical row, never more than three.
//   3. every wave counts the entries of its part above and at the k-th key; the counts of the waves before it
//      are its offsets.  Taken entries get their place in index order from ballots; ties at the k-th value
//      go to the LOWER index.
//   4. optionally (k <= kTopkSortMax) the order by descending value, ties by ascending index, of 64-bit
//      (key, ~index) words: counted in 2048 bins that span them, each word's place then is the number of words in higher
//      bins plus those of its own bin that are larger (four barriers, about one comparison per word).  Up to a
//      wave of words, and where more than 64 share a bin (ties, a few outliers in several parts of the row), a bitonic
//      sort: exchanges over less than a wave's elements are DPP and lane swaps in registers, only the wider ones go through
//      LDS.  Its 55 steps on 1024 words were 4 us of the 15, all VALU work of a single compute unit.
// Measured (with shuffles in place of the DPP scans, 1 us more), sorted, B 4, bitonic sort -> counting: S 8192, k 128 11.1 -> 10.1 us, 512 13.0 -> 10.8, 1024 14.9 -> 11.3,
// 4096 31.0 -> 17.0; S 32768, k 2048 32.1 -> 26.5; S 131072, k 4096 103.8 -> 94.1.  k 64 is equal either way.  Rows with a
// crowded bin pay for the count and the sort (S 8192, k 1024, 16.0 -> 16.8).
// The threshold form is step 3 alone with a given threshold.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "flash_colsum.h"
#include "fcs_device.h"
#include "fcs_kernels.h"

namespace fcs {

namespace {

constexpr int kTopkSortMax = FCS_TOPK_SORT_MAX;
constexpr int kTopkThreads = 1024;
constexpr int kTopkWaves = kTopkThreads / 64;
constexpr int kTopkBins = 2048;      // two per thread
constexpr int kTopkBinBits = 11;
constexpr int kTopkMaxRegs = 32;     // elements per lane that stay in registers
constexpr int kTopkCountMin = 64;    // more than this many are ordered by counting
constexpr int kTopkCrowd = 64;       // ... if no bin holds more than this many of them

// monotone map float -> uint32: a < b  <=>  key(a) < key(b)  (-0 < +0, NaNs at the two ends)
__device__ __forceinline__ uint32_t order_key(float v)
{
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float key_value(uint32_t key)  // its inverse
{
    return __builtin_bit_cast(float, (key & 0x80000000u) ? (key & 0x7fffffffu) : ~key);
}

// This wave's part of a row: elements first + 64 j + lane for j < n_j, E of them in registers (E = 0: read again
// by every sweep).  CANON: -0 counts as +0 (the value comparison `>=` of the threshold form, not the bit order
// of top-k).
template <int E, bool CANON>
struct RowPart {
    static constexpr int kBatch = 8;
    const float *row;
    int S, first, n_j;
    uint32_t keys[E > 0 ? E : 1];

    __device__ __forceinline__ static uint32_t key_at(const float *p, int i, int n)  // of p[i], or of 0 past its n entries
    {
        const float v = (i < n) ? p[i] : 0.f;
        return order_key(CANON ? v + 0.0f : v);
    }
    __device__ __forceinline__ void init(const float *r, int n, int wave, int lane)
    {
        row = r;
        S = n;
        n_j = (E > 0) ? E : ((n - 1) / (kBatch * kTopkThreads) + 1) * kBatch;
        first = wave * n_j * 64 + lane;
        if constexpr (E > 0) {
#pragma unroll
            for (int j = 0; j < E; ++j) keys[j] = key_at(row, first + 64 * j, S);
        }
    }
    // f(index, key, exists) for every element of the lane, in ascending order; all lanes of the wave together
    template <typename F>
    __device__ __forceinline__ void each(F f) const
    {
        if constexpr (E > 0) {
            int at = first;
            asm volatile("" : "+v"(at));  // every sweep forms its own comparisons: kept masks would spill
#pragma unroll
            for (int j = 0; j < E; ++j) f(at + 64 * j, keys[j], at + 64 * j < S);
        } else {
            // The batch's start is wave-uniform and unsigned (a row's length rounded up to whole sweeps may pass 2^31); its
            // entries are addressed from there.
            const int lane = threadIdx.x & 63;
            uint32_t base = (uint32_t)__builtin_amdgcn_readfirstlane(first - lane);
            for (int j0 = 0; j0 < n_j; j0 += kBatch, base += 64 * kBatch) {
                const int left = (base < (uint32_t)S) ? (int)min((uint32_t)S - base, 64u * kBatch) : 0;
                const float *p = row + base;
                uint32_t k[kBatch];  // that many loads in flight
#pragma unroll
                for (int j = 0; j < kBatch; ++j) k[j] = key_at(p, 64 * j + lane, left);
#pragma unroll
                for (int j = 0; j < kBatch; ++j) f((int)(base + 64 * j + lane), k[j], 64 * j + lane < left);
            }
        }
    }
};

struct TopkLds {
    int hist[kTopkBins];
    int wsum[kTopkWaves];
    uint32_t wmin[kTopkWaves], wmax[kTopkWaves];
    int2 wcnt[kTopkWaves];
    int bin, above, count;
    int crowded;
};

// A wave's running totals op(v of lane 0, .., v of this lane), in registers: within rows of 16 lanes, then the rows' last lanes to the
// rows above (a lane without a partner takes `none`).  A step is one DPP instruction, where a shuffle is an LDS round trip.  us per
// selection, shuffles -> this: B 4, S 8192, k 1024 11.4 -> 10.4, S 1898, k 314 8.0 -> 6.8, S 32768, k 2048 26.0 -> 24.7.
template <typename F>
__device__ __forceinline__ uint32_t lanes_below(uint32_t v, uint32_t none, F op)
{
#define FCS_SCAN_STEP(CTRL, ROWS) v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)none, (int)v, CTRL, ROWS, 0xF, false))
    FCS_SCAN_STEP(0x111, 0xF);  // row_shr:1
    FCS_SCAN_STEP(0x112, 0xF);
    FCS_SCAN_STEP(0x114, 0xF);
    FCS_SCAN_STEP(0x118, 0xF);
    FCS_SCAN_STEP(0x142, 0xA);  // row_bcast:15, into rows 1 and 3
    FCS_SCAN_STEP(0x143, 0xC);  // row_bcast:31, into rows 2 and 3
#undef FCS_SCAN_STEP
    return v;
}
__device__ __forceinline__ uint32_t last_lane(uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, 63); }

// How many of the counted keys lie in the bins of higher threads; c: those in this thread's two.  One barrier.
__device__ __forceinline__ int in_higher_bins(int c, TopkLds &lds, int wave, int lane)
{
    const uint32_t run = lanes_below((uint32_t)c, 0u, [](uint32_t a, uint32_t b) { return a + b; }), all = last_lane(run);
    if (lane == 0) lds.wsum[wave] = (int)all;
    __syncthreads();
    int above = (int)(all - run);
#pragma unroll
    for (int w = 0; w < kTopkWaves; ++w) above += (w > wave) ? lds.wsum[w] : 0;
    return above;
}

// Places of the taken elements in index order.  thr: elements with a larger key are taken, and the first `need`
// with an equal one.  put(place, index, key) is called for each; returns their number (block-uniform).  One barrier.
template <int E, bool CANON, typename Put>
__device__ __forceinline__ int take_in_order(const RowPart<E, CANON> &part, uint32_t thr, int need, TopkLds &lds, int wave, int lane,
                                             Put put)
{
    int gt_n = 0, eq_n = 0;  // wave-uniform
    part.each([&](int, uint32_t key, bool in) {
        gt_n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(in && key > thr));
        eq_n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(in && key == thr));
    });
    if (lane == 0) lds.wcnt[wave] = int2{gt_n, eq_n};
    __syncthreads();
    int gt = 0, eq = 0, gt_all = 0, eq_all = 0;  // above / at the threshold before this wave's part, and in the row
#pragma unroll
    for (int w = 0; w < kTopkWaves; ++w) {
        const int2 c = lds.wcnt[w];
        gt += (w < wave) ? c.x : 0;
        eq += (w < wave) ? c.y : 0;
        gt_all += c.x;
        eq_all += c.y;
    }
    const uint64_t below = (1ull << lane) - 1ull;
    asm volatile("" : "+v"(thr));
    part.each([&](int i, uint32_t key, bool in) {
        const bool is_gt = in && key > thr, is_eq = in && key == thr;
        const uint64_t bg = __builtin_amdgcn_ballot_w64(is_gt), be = __builtin_amdgcn_ballot_w64(is_eq);
        const int eq_before = eq + __builtin_popcountll(be & below);
        if (is_gt || (is_eq && eq_before < need)) put(gt + __builtin_popcountll(bg & below) + min(eq_before, need), i, key);
        gt += __builtin_popcountll(bg);
        eq += __builtin_popcountll(be);
    });
    return gt_all + min(eq_all, need);
}

// the value of lane (lane ^ MASK)
template <int MASK>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v, int lane)
{
    auto dpp = [](uint32_t x, auto ctrl) {
        return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, decltype(ctrl)::value, 0xF, 0xF, false);
    };
    if constexpr (MASK == 1) return dpp(v, std::integral_constant<int, kDppXor1>{});
    else if constexpr (MASK == 2) return dpp(v, std::integral_constant<int, kDppXor2>{});
    else if constexpr (MASK == 4)  // l ^ 7, then ^ 3
        return dpp(dpp(v, std::integral_constant<int, kDppHalfMirror>{}), std::integral_constant<int, 0x1B>{});
    else if constexpr (MASK == 8) return dpp(v, std::integral_constant<int, 0x128>{});  // rotate a row of 16 by 8
    else {
        // the swap leaves, of two copies, the partner's value in one of them: which one depends on the half
        uint32_t x = v, y = v;
        if constexpr (MASK == 16) asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
        else asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(x), "+v"(y));
        return (lane & MASK) ? x : y;
    }
}

// Bitonic sort, largest first, of n2 (a power of two, at most 1024 SE) 64-bit words in buf[0 .. n2); thread t holds
// the words t SE .. t SE + SE - 1.  buf has two halves of kTopkSortMax words: an exchange through LDS writes one and
// the next such exchange the other, so that each costs one barrier.  Every thread of the block calls it; the result
// stays in `w`.
template <int SE>
__device__ __forceinline__ void sort_descending(uint64_t *buf, int n2, int tid, uint64_t (&w)[SE])
{
    const int lane = tid & 63;
#pragma unroll
    for (int s = 0; s < SE; ++s) w[s] = (tid * SE + s < n2) ? buf[tid * SE + s] : 0;
    int half = 1;
    // keep the larger word where the element comes first of its pair in a block that ends up descending
    auto keep = [&](uint64_t mine, uint64_t other, int e, int stride, int size) {
        const bool larger = ((e & stride) == 0) == ((e & size) == 0);
        return ((mine > other) == larger) ? mine : other;
    };
    auto in_wave = [&](auto mask_c, int size) {
        constexpr int MASK = decltype(mask_c)::value;
#pragma unroll
        for (int s = 0; s < SE; ++s) {
            const uint32_t lo = lane_xor<MASK>((uint32_t)w[s], lane), hi = lane_xor<MASK>((uint32_t)(w[s] >> 32), lane);
            w[s] = keep(w[s], ((uint64_t)hi << 32) | lo, tid * SE + s, MASK * SE, size);
        }
    };
    for (int size = 2; size <= n2; size <<= 1) {
        int stride = size >> 1;
        for (; stride >= 64 * SE; stride >>= 1) {
            uint64_t *b = buf + half * kTopkSortMax;
            half ^= 1;
#pragma unroll
            for (int s = 0; s < SE; ++s)
                if (tid * SE + s < n2) b[tid * SE + s] = w[s];
            __syncthreads();
#pragma unroll
            for (int s = 0; s < SE; ++s)
                if (tid * SE + s < n2) w[s] = keep(w[s], b[(tid * SE + s) ^ stride], tid * SE + s, stride, size);
        }
        if (stride >= 32 * SE) in_wave(std::integral_constant<int, 32>{}, size);
        if (stride >= 16 * SE) in_wave(std::integral_constant<int, 16>{}, size);
        if (stride >= 8 * SE) in_wave(std::integral_constant<int, 8>{}, size);
        if (stride >= 4 * SE) in_wave(std::integral_constant<int, 4>{}, size);
        if (stride >= 2 * SE) in_wave(std::integral_constant<int, 2>{}, size);
        if (stride >= SE) in_wave(std::integral_constant<int, 1>{}, size);
#pragma unroll
        for (int st = SE / 2; st > 0; st >>= 1) {
            if (stride >= st) {
#pragma unroll
                for (int s = 0; s < SE; ++s)
                    if ((s & st) == 0) {
                        const uint64_t a = w[s], b = w[s + st];
                        w[s] = keep(a, b, tid * SE + s, st, size);
                        w[s + st] = keep(b, a, tid * SE + s + st, st, size);
                    }
            }
        }
    }
}

// The same order by counting, for k words in buf[0 .. k) whose keys are lo or more and are counted in lds.hist by
// count_bin: every word goes to its bin's part of buf's second half, takes its place from the words of its bin that
// are larger (all words differ, so the places do not depend on the order in which a bin was filled), and buf[0 .. k) ends up
// in order.  False, with buf as it was, where a bin is crowded: a word is compared with all of its bin.  Block-uniform.
__device__ __forceinline__ int count_bin(uint32_t key, uint32_t lo, int shift)
{
    return (int)min((key - lo) >> shift, (uint32_t)(kTopkBins - 1));
}
template <int SE>
__device__ __forceinline__ bool count_descending(uint64_t *buf, int k, uint32_t lo, int shift, TopkLds &lds, int tid, int wave, int lane)
{
    const int c0 = lds.hist[2 * tid], c1 = lds.hist[2 * tid + 1];
    if (max(c0, c1) > kTopkCrowd) lds.crowded = 1;
    const int above = in_higher_bins(c0 + c1, lds, wave, lane);
    if (lds.crowded) return false;
    lds.hist[2 * tid + 1] = above;  // where a bin's words begin; where they end once they are all in
    lds.hist[2 * tid] = above + c1;
    __syncthreads();
    uint64_t w[SE], *binned = buf + kTopkSortMax;
#pragma unroll
    for (int s = 0; s < SE; ++s) {
        const int i = tid + s * kTopkThreads;
        w[s] = (i < k) ? buf[i] : 0;
        if (i < k) binned[atomicAdd(&lds.hist[count_bin((uint32_t)(w[s] >> 32), lo, shift)], 1)] = w[s];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < SE; ++s) {
        if (tid + s * kTopkThreads < k) {
            const int bin = count_bin((uint32_t)(w[s] >> 32), lo, shift), end = lds.hist[bin];
            const int start = (bin + 1 < kTopkBins) ? lds.hist[bin + 1] : 0;
            int place = start;
            for (int j = start; j < end; ++j) place += (binned[j] > w[s]) ? 1 : 0;
            buf[place] = w[s];
        }
    }
    __syncthreads();
    return true;
}

}  // namespace

template <int E>
__global__ __launch_bounds__(kTopkThreads) void fcs_topk_kernel(const float *means, int S, int k, int64_t *idx_out, float *val_out,
                                                                int sorted)
{
    __shared__ TopkLds lds;
    __shared__ uint64_t buf[2 * kTopkSortMax];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int64_t *io = idx_out + (int64_t)blockIdx.x * k;
    float *vo = val_out ? val_out + (int64_t)blockIdx.x * k : nullptr;
    RowPart<E, false> part;
    part.init(means + (int64_t)blockIdx.x * S, S, wave, lane);

    // ---- 1. range of the row's keys
    uint32_t kmin = 0xffffffffu, kmax = 0;
    part.each([&](int, uint32_t key, bool in) {
        kmin = in ? min(kmin, key) : kmin;
        kmax = in ? max(kmax, key) : kmax;
    });
    kmin = last_lane(lanes_below(kmin, 0xffffffffu, [](uint32_t a, uint32_t b) { return min(a, b); }));
    kmax = last_lane(lanes_below(kmax, 0u, [](uint32_t a, uint32_t b) { return max(a, b); }));
    if (lane == 0) {
        lds.wmin[wave] = kmin;
        lds.wmax[wave] = kmax;
    }
    lds.hist[2 * tid] = lds.hist[2 * tid + 1] = 0;
    if (tid == 0) lds.crowded = 0;
    __syncthreads();
    uint32_t kmax2 = 0;  // of the waves' largest keys the second
    kmax = 0;
#pragma unroll
    for (int w = 0; w < kTopkWaves; ++w) {
        const uint32_t v = lds.wmax[w];
        kmin = min(kmin, lds.wmin[w]);
        kmax2 = max(kmax2, min(kmax, v));
        kmax = max(kmax, v);
    }

    // ---- 2. the k-th largest key lies in [lo, lo + span]; `want` is its rank (1 = largest) among the keys in there.
    // Afterwards: keys above `lo` are taken, and the first `want` that equal it
    uint32_t lo = kmin, span = kmax - kmin;
    int want = k;
    while (span != 0) {  // block-uniform
        const int bits = 32 - __builtin_clz(span), shift = max(0, bits - kTopkBinBits);
        part.each([&](int, uint32_t key, bool in) {
            const uint32_t off = key - lo;  // wraps for keys below lo
            if (in && off <= span) atomicAdd(&lds.hist[off >> shift], 1);
        });
        __syncthreads();
        // bins 2 tid and 2 tid + 1; suffix sums over the threads
        const int c0 = lds.hist[2 * tid], c1 = lds.hist[2 * tid + 1];
        const int above = in_higher_bins(c0 + c1, lds, wave, lane);
        if (above < want && want <= above + c1) {
            lds.bin = 2 * tid + 1;
            lds.above = above;
            lds.count = c1;
        } else if (above + c1 < want && want <= above + c1 + c0) {
            lds.bin = 2 * tid;
            lds.above = above + c1;
            lds.count = c0;
        }
        lds.hist[2 * tid] = lds.hist[2 * tid + 1] = 0;
        __syncthreads();
        want -= lds.above;
        const uint32_t bin_lo = lo + ((uint32_t)lds.bin << shift);
        const uint32_t bin_hi_off = ((uint32_t)lds.bin << shift) + ((1u << shift) - 1u);
        span = min(bin_hi_off, span) - ((uint32_t)lds.bin << shift);  // the last bin may be cut off
        lo = bin_lo;
        if (want == lds.count) {  // the bin is taken whole: every key from its lower end on
            want = S;
            break;
        }
    }

    // ---- 3. and 4.
    if (!sorted || k > kTopkSortMax) {
        take_in_order(part, lo, want, lds, wave, lane, [&](int place, int i, uint32_t key) {
            if (place < k) {
                io[place] = i;
                if (vo) vo[place] = key_value(key);
            }
        });
        return;
    }
    int n2 = 1;
    while (n2 < k) n2 <<= 1;
    // zero words sort behind every real one (whose lower half is the complement of an index)
    for (int i = k + tid; i < n2; i += kTopkThreads) buf[i] = 0;
    const bool equal = kmax == lo;  // all that are taken: in order as they are
    const bool count = k > kTopkCountMin && !equal;
    // The bins span the taken keys, or without those of one wave where these (a context's first tokens) would leave the
    // others an eighth of the bins: they meet in the last one.
    const uint32_t top = (kmax2 > lo && (kmax - lo) >> 3 > kmax2 - lo) ? kmax2 : kmax;
    const int shift = (top == lo) ? 0 : max(0, 32 - __builtin_clz(top - lo) - kTopkBinBits);
    take_in_order(part, lo, want, lds, wave, lane, [&](int place, int i, uint32_t key) {
        if (place < k) {
            buf[place] = ((uint64_t)key << 32) | (uint32_t)~i;
            if (count) atomicAdd(&lds.hist[count_bin(key, lo, shift)], 1);
        }
    });
    __syncthreads();
    auto put = [&](int e, uint64_t w) {
        io[e] = (int)~(uint32_t)w;
        if (vo) vo[e] = key_value((uint32_t)(w >> 32));
    };
    auto finish = [&](auto se_c) {
        constexpr int SE = decltype(se_c)::value;
        if (equal || (count && count_descending<SE>(buf, k, lo, shift, lds, tid, wave, lane))) {
            for (int e = tid; e < k; e += kTopkThreads) put(e, buf[e]);
            return;
        }
        uint64_t w[SE];
        sort_descending<SE>(buf, n2, tid, w);
#pragma unroll
        for (int s = 0; s < SE; ++s)
            if (tid * SE + s < k) put(tid * SE + s, w[s]);
    };
    if (n2 <= kTopkThreads) finish(std::integral_constant<int, 1>{});
    else if (n2 <= 2 * kTopkThreads) finish(std::integral_constant<int, 2>{});
    else finish(std::integral_constant<int, 4>{});
    static_assert(kTopkSortMax <= 4 * kTopkThreads, "words per thread above");
}

template <int E>
__global__ __launch_bounds__(kTopkThreads) void fcs_threshold_kernel(const float *means, int S, float tau, int64_t *idx_out,
                                                                     int32_t *count_out)
{
    __shared__ TopkLds lds;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    RowPart<E, true> part;
    part.init(means + (int64_t)blockIdx.x * S, S, wave, lane);
    int64_t *io = idx_out + (int64_t)blockIdx.x * S;
    // value >= tau  <=>  key(value) >= key(tau) once -0 is read as +0 on both sides (the bit order alone puts
    // -0 below +0): "larger than thr, or equal to thr with unlimited ties" with thr = key(tau + 0)
    const int n = take_in_order(part, order_key(tau + 0.0f), S, lds, wave, lane, [&](int place, int i, uint32_t) { io[place] = i; });
    if (threadIdx.x == 0) count_out[blockIdx.x] = n;
}

// Elements per lane for rows of S entries: the smallest power of two that holds the row in registers, 0 (re-read)
// beyond kTopkMaxRegs.
template <typename F>
static void with_row_regs(int S, F f)
{
    const int e = (S - 1) / kTopkThreads + 1;
    if (e <= 1) f(std::integral_constant<int, 1>{});
    else if (e <= 2) f(std::integral_constant<int, 2>{});
    else if (e <= 4) f(std::integral_constant<int, 4>{});
    else if (e <= 8) f(std::integral_constant<int, 8>{});
    else if (e <= 16) f(std::integral_constant<int, 16>{});
    else if (e <= kTopkMaxRegs) f(std::integral_constant<int, kTopkMaxRegs>{});
    else f(std::integral_constant<int, 0>{});
}

}  // namespace fcs

extern "C" {

int fcs_topk_f32(const float *means, int B, int S, int k, int64_t *idx_out, float *val_out, int sorted, void *hip_stream)
{
    if (!means || !idx_out) return FCS_E_NULL;
    if (B < 1 || S < 1 || k < 1 || k > S) return FCS_E_DIMS;
    if (sorted && k > FCS_TOPK_SORT_MAX) return FCS_E_DIMS;
    fcs::with_row_regs(S, [&](auto e) {
        hipLaunchKernelGGL(fcs::fcs_topk_kernel<decltype(e)::value>, dim3(B), dim3(fcs::kTopkThreads), 0,
                           reinterpret_cast<hipStream_t>(hip_stream), means, S, k, idx_out, val_out, sorted ? 1 : 0);
    });
    return (int)hipGetLastError();
}

int fcs_threshold_f32(const float *means, int B, int S, float tau, int64_t *idx_out, int32_t *count_out, void *hip_stream)
{
    if (!means || !idx_out || !count_out) return FCS_E_NULL;
    if (B < 1 || S < 1) return FCS_E_DIMS;
    if (tau != tau) return FCS_E_SCALE;
    fcs::with_row_regs(S, [&](auto e) {
        hipLaunchKernelGGL(fcs::fcs_threshold_kernel<decltype(e)::value>, dim3(B), dim3(fcs::kTopkThreads), 0,
                           reinterpret_cast<hipStream_t>(hip_stream), means, S, tau, idx_out, count_out);
    });
    return (int)hipGetLastError();
}

}  // extern "C"
