// Attention column means on gfx950 (MI355X): launch order of the paths and the final reduction.
//
//   pass 1 (fcs_rowstream_kernel, fcs_stream_kernels.h)  per row (m, log2 l) with
//          l = sum_j 2^((s_ij - m) * c), c = scale*log2(e), or (m, l) per part of a row block.
//   pass 2 (fcs_colstream_kernel, fcs_stream_kernels.h)  column sums of 2^((s_ij - m_i) * c - log2 l_i),
//          one partial slab per workgroup and key chunk that its share touches.
//   fcs_finalize_kernel (here) adds the slabs in a fixed order: no atomics anywhere, every
//          partial has exactly one writer.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <stdio.h>

#include "fcs_device.h"
#include "fcs_kernels.h"

namespace fcs {

// slab lanes for n slabs: the fewest of 8, 16, 32 that leave a lane at most four slabs (32 beyond 128 slabs)
static inline int slab_lanes(int n) { return n <= 32 ? 8 : n <= 64 ? 16 : 32; }

// The summation tree of one output over n slabs with SL slab lanes: lane sl adds the slabs sl, sl + SL,
// sl + 2 SL, ... in index order into four running sums (slab sl + j SL goes to sum j % 4, so four loads
// are in flight), and its total is (s0 + s1) + (s2 + s3).  `stride` is the distance between slabs in floats.
template <int SL>
__device__ __forceinline__ float slab_lane_total(const float *p, int64_t stride, int n, int sl)
{
    float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
    for (int gi = sl; gi < n; gi += 4 * SL) {
        s0 += p[(int64_t)gi * stride];
        if (gi + SL < n) s1 += p[(int64_t)(gi + SL) * stride];
        if (gi + 2 * SL < n) s2 += p[(int64_t)(gi + 2 * SL) * stride];
        if (gi + 3 * SL < n) s3 += p[(int64_t)(gi + 3 * SL) * stride];
    }
    return (s0 + s1) + (s2 + s3);
}

// out = inv_norm * (partial[0] + partial[1] + ...).  A block owns 32 consecutive outputs; its
// SL slab lanes each add every SL-th slab in index order (four running sums, so that four loads
// are in flight per thread) and the SL sub-totals are then added in lane order: the summation
// tree is fixed by (number of slabs, SL), i.e.
// bit-reproducible, while SL x 4 loads per output are in flight instead of one.  SL = 8 for the
// usual few dozen slabs, 16 or 32 for more (slab_lanes()): a small batch can leave hundreds of
// slabs per batch entry (B 1, H 16, S 1024 on the fused path: 512 slabs of 1024 outputs, where 8
// lanes took longer than the kernel that wrote the slabs).
//
// SHARES (two-pass path): a key chunk has one slab per workgroup of the column pass whose share of the line touches it,
// as many as its units take; the slabs of all chunks lie one behind the other.
template <int SL, bool SHARES>
__global__ __launch_bounds__(32 * SL) void fcs_finalize_kernel(const Args a)
{
    __shared__ float sub[SL][32];
    fetch_args(a);
    const int64_t n = (int64_t)a.B * a.Sk;
    const int col = threadIdx.x & 31, sl = threadIdx.x >> 5;
    const int64_t idx = (int64_t)blockIdx.x * 32 + col;
    float v = 0.f;
    if (idx < n) {
        if constexpr (SHARES) {
            const int b = (int)((n >> 32) == 0 ? (uint32_t)idx / (uint32_t)a.Sk : idx / a.Sk);
            int in_chunk;
            const int cx = a.c_by_chunk.quot((int)(idx - (int64_t)b * a.Sk), in_chunk);
            const int pairs = a.c_line.pairs(a.c_nrb, a.c_cs, cx, a.c_every), at = a.c_line.sum(a.c_nrb, cx * a.c_cs);
            const int before = at + pairs * a.c_line.start;
            const int len = (a.c_line.sum(a.c_nrb, (cx + 1) * a.c_cs) - at + a.c_line.sees(a.c_nrb, a.c_cs, cx) * a.c_line.start) * a.v_heads;
            const int start = b * (int)a.c_by_batch.d + before * a.v_heads, w0 = a.c_by_seg.quot(start + a.c_line.start);
            const int slabs = (len > 0) ? a.c_by_seg.quot(start + len - 1) - w0 + 1 : 0;  // 0: no row sees the chunk
            const float *p = a.partial + (w0 + (int64_t)b * a.c_nchunks + cx) * a.c_chunk + in_chunk;
            v = slab_lane_total<SL>(p, a.c_chunk, slabs, sl);
        } else {
            v = slab_lane_total<SL>(a.partial + idx, n, a.n_partials, sl);
        }
    }
    sub[sl][col] = v;
    __syncthreads();
    if (sl == 0 && idx < n) {
        float t = sub[0][col];
#pragma unroll
        for (int j = 1; j < SL; ++j) t += sub[j][col];
        a.out[idx] = t * a.inv_norm;
        if (a.out_h) a.out_h[idx] = (_Float16)(t * a.inv_norm);
    }
}

// ------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------
template <bool SHARES>
static hipError_t launch_finalize_t(const Args &a, hipStream_t st)
{
    const int64_t n = (int64_t)a.B * a.Sk;
    const dim3 grid((unsigned)((n + 31) / 32));
    switch (slab_lanes(a.n_partials)) {
    case 32: hipLaunchKernelGGL((fcs_finalize_kernel<32, SHARES>), grid, dim3(1024), 0, st, a); break;
    case 16: hipLaunchKernelGGL((fcs_finalize_kernel<16, SHARES>), grid, dim3(512), 0, st, a); break;
    default: hipLaunchKernelGGL((fcs_finalize_kernel<8, SHARES>), grid, dim3(256), 0, st, a); break;
    }
    return hipGetLastError();
}

hipError_t launch_finalize(const Args &a, hipStream_t st) { return launch_finalize_t<false>(a, st); }

size_t describe_finalize(const Args &a, bool shares, char *buf, size_t n)
{
    const int r = snprintf(buf, n, " + fcs_finalize_kernel<%d%s> grid %lld", slab_lanes(a.n_partials), shares ? ",true" : "",
                           (long long)(((int64_t)a.B * a.Sk + 31) / 32));
    return r < 0 ? 0 : (size_t)r;
}

// the two-pass path: row statistics, column sums (which also merge the key splits), final reduction
static hipError_t launch_two_pass(const Plan &p, const Args &a, hipStream_t st)
{
    hipError_t e = launch_rowstream(p, a, st);
    if (e != hipSuccess) return e;
    e = launch_colstream(p, a, st);
    if (e != hipSuccess) return e;
    return p.c_direct ? hipSuccess : launch_finalize_t<true>(a, st);
}

int launch_colsum(const Plan &p, const Args &a, void *stream)
{
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (p.fewrows) return (int)launch_fewrows(p, a, st);
    if (p.small) return (int)launch_small(p, a, st);
    if (p.tall) return (int)launch_tall(p, a, st);
    if (p.fused) return (int)launch_fused(p, a, st);
    return (int)launch_two_pass(p, a, st);
}

size_t describe_colsum(const Plan &p, const Args &a, char *buf, size_t n)
{
    if (p.fewrows) return describe_fewrows(p, a, buf, n);
    if (p.small) return describe_small(p, a, buf, n);
    if (p.tall) return describe_tall(p, a, buf, n);
    if (p.fused) return describe_fused(p, a, buf, n);
    return describe_two_pass(p, a, buf, n);
}

}  // namespace fcs
