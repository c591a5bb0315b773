// Two-pass path: which kernels a plan launches.  Kernels and their launchers: fcs_stream_kernels.h.
#include <stdio.h>

#include "fcs_stream_kernels.h"

namespace fcs {

extern template hipError_t launch_rowstream_f<false>(const Plan &, const Args &, hipStream_t);
extern template hipError_t launch_rowstream_f<true>(const Plan &, const Args &, hipStream_t);
extern template hipError_t launch_colstream_f<false>(const Plan &, const Args &, hipStream_t);
extern template hipError_t launch_colstream_f<true>(const Plan &, const Args &, hipStream_t);

size_t describe_two_pass(const Plan &p, const Args &a, char *buf, size_t n)
{
    const bool pre = stream_prescaled(p, a);
    const int nb1 = p.qw / 32;
    const char *fold = p.fold > 1 ? ",true" : "";  // query heads of a key head in one unit
    int r = snprintf(buf, n,
                     "fcs_rowstream_kernel<%d,%d,%d,%s,%s%s> grid %d x %d x %d + fcs_colstream_kernel<%d,%d,%d,%s,%s%s> grid %d x %d x %d, "
                     "%d units per workgroup",
                     p.Dp, nb1, p.k1_waves, p.bf16 ? "true" : "false", pre ? "true" : "false", fold, p.n_qblk, p.n_chunks, p.B * p.v_heads, p.Dp,
                     p.c_nb, p.c_waves, p.bf16 ? "true" : "false", pre ? "true" : "false", fold, p.c_nchunks, p.c_groups, p.B, p.c_upg);
    if (r < 0) return 0;
    const size_t len = (size_t)r;
    if (p.c_groups > 1) return len + describe_finalize(a, len < n ? buf + len : nullptr, len < n ? n - len : 0);
    return len;
}

hipError_t launch_rowstream(const Plan &p, const Args &a, hipStream_t st)
{
    return p.fold > 1 ? launch_rowstream_f<true>(p, a, st) : launch_rowstream_f<false>(p, a, st);
}

hipError_t launch_colstream(const Plan &p, const Args &a, hipStream_t st)
{
    return p.fold > 1 ? launch_colstream_f<true>(p, a, st) : launch_colstream_f<false>(p, a, st);
}

}  // namespace fcs
