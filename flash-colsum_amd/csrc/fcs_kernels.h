// Kernel argument block and the single launch entry used by the C ABI layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fcs_plan.h"

namespace fcs {

struct Args {
    const _Float16 *q;
    const _Float16 *k;
    int64_t qs_b, qs_h, qs_s;  // element strides (last dim is 1)
    int64_t ks_b, ks_h, ks_s;
    int B, H, Sq, Sk;
    int D;               // head dim of the tensors (a multiple of 8); kernels compiled for a wider head read zeros beyond it
    int kv_group;        // query heads per key head (1 unless grouped-query): key head = head / kv_group
    uint32_t kv_magic;   // ceil(2^32 / kv_group), for the division above (unused when kv_group == 1)
    int q_rows;          // query rows that are averaged
    // two-pass path: the averaged rows as its kernels number them.  fold == 1: row v of head h is query row v.  fold > 1:
    // the `fold` query heads of a key head form one head of v_rows = fold * q_rows rows (then kv_group is 1)
    int fold, v_heads, v_rows;
    uint32_t fold_magic;  // ceil(2^31 / q_rows), for v / q_rows (unused when fold == 1)
    int causal, k_past;  // key j visible to query i  <=>  j <= k_past + i
    int pre_end;         // two-pass path, pre-scaled variant: the 64-key stages that end at or below this key (a multiple
                         // of 64) run on Q * c rounded to fp16 in both passes; the keys that every averaged row sees
    int negate;          // scale < 0: scores are negated by flipping the stationary operand's sign
    float c;             // |scale| * log2(e)
    // pass 1
    StageLine r_line;  // the stages of its row blocks in units of r_unit; workgroup w takes [w * r_seg, (w + 1) * r_seg) of all r_len
    int r_unit, r_seg, r_len, r_blocks, r_whole, n_qblk;
    FastDiv r_by_seg, r_by_head, r_by_block, by_heads;
    float2 *stat;  // r_whole: [B*v_heads * n_qblk][rows of a block] (m, log2 l): row maximum in score units (0 on the
                   //          unstabilised path) and log2 of sum_j 2^((s_ij - m) * c)
                   // else:    set w + i holds (m, l) of share w's part of row block i (i = head * n_qblk + block); an
                   //          empty part is (0, 0)
    // pass 2
    int c_chunk, c_nchunks, c_nrb;  // keys per chunk, chunks, row blocks per head
    StageLine c_line;               // the stages of its units, as for pass 1; chunk after chunk
    int c_unit, c_cs, c_seg, c_len, c_blocks, c_direct, c_every;  // c_cs: units per chunk
    FastDiv c_by_seg, c_by_batch, c_by_chunks, c_by_chunk, c_by_blocks;
    float *partial;  // slabs; two-pass path: [..][c_chunk], slab w + i is share w's of chunk i (i = batch entry * c_nchunks + chunk)
    float *out;      // [B][Sk]
    _Float16 *out_h; // [B][Sk] or nullptr: the same means rounded to fp16
    float inv_norm;  // 1 / (H * q_rows)
    int n_partials;  // slabs of `partial` that fcs_finalize_kernel adds up
    // fused single-kernel path (scores stay in registers)
    int f_kg;        // waves along the key axis (1, 2, 4 or 8); 8 / f_kg waves along the query axis
    int f_tpw;       // 32-key tiles per wave (<= 8)
    int f_nqblk;     // blocks along the query axis (32 * 8 / f_kg rows each; short-sequence path: 32-row tiles per head)
    int f_hpg;       // heads per block
    int f_rbpw;      // adjacent row blocks per block (a block walks over f_rbpw x f_hpg units)
    int f_nwgq;      // blocks along the query axis: ceil(f_nqblk / f_rbpw)
    int f_hg;        // head groups (fused and few-rows paths): a batch entry has f_hg * f_nwgq workgroups
};

#if defined(__HIP_DEVICE_COMPILE__) || defined(__HIPCC__)
// First thing in a kernel: one word of every 64 bytes of its arguments, requested together.  The compiler loads arguments
// where they are first used, and each of those loads would wait for a line of its own to come from memory, one after the
// other; behind this they hit the scalar cache.
__device__ __forceinline__ void fetch_args(const Args &a)
{
    const int *w = reinterpret_cast<const int *>(&a);
    constexpr int N = (int)(sizeof(Args) / sizeof(int));
    static_assert(N > 80 && N <= 96, "one word of each line");
    asm volatile("" ::"s"(w[0]), "s"(w[16]), "s"(w[32]), "s"(w[48]), "s"(w[64]), "s"(w[80]), "s"(w[N - 1]));
}
#endif

// Enqueues every kernel of one call on `stream`; returns 0 or the hipError_t of a failed launch.
int launch_colsum(const Plan &p, const Args &a, void *stream);

// fused path, defined in fcs_fused.hip, and (p.tall) fcs_tall.hip
hipError_t launch_fused(const Plan &p, const Args &a, hipStream_t st);
hipError_t launch_tall(const Plan &p, const Args &a, hipStream_t st);
// few-rows path (fcs_fewrows.hip): p.fewrows == 1
hipError_t launch_fewrows(const Plan &p, const Args &a, hipStream_t st);
// short-sequence path (fcs_small.hip): p.small == 1
hipError_t launch_small(const Plan &p, const Args &a, hipStream_t st);

// row-statistics pass and column pass of the two-pass path (fcs_stream_kernels.h)
hipError_t launch_rowstream(const Plan &p, const Args &a, hipStream_t st);
hipError_t launch_colstream(const Plan &p, const Args &a, hipStream_t st);

// shared final reduction out = inv_norm * sum of the n_partials slabs (fcs_kernels.hip)
hipError_t launch_finalize(const Args &a, hipStream_t st);

// Text description of what launch_colsum(p, a, .) launches; snprintf semantics.
size_t describe_colsum(const Plan &p, const Args &a, char *buf, size_t n);
size_t describe_fused(const Plan &p, const Args &a, char *buf, size_t n);
size_t describe_tall(const Plan &p, const Args &a, char *buf, size_t n);
size_t describe_fewrows(const Plan &p, const Args &a, char *buf, size_t n);
size_t describe_small(const Plan &p, const Args &a, char *buf, size_t n);
size_t describe_two_pass(const Plan &p, const Args &a, char *buf, size_t n);
size_t describe_finalize(const Args &a, bool shares, char *buf, size_t n);

}  // namespace fcs
