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
    const char *bf = p.bf16 ? "true" : "false", *ps = pre ? "true" : "false";
    // the kernels' last argument, ONE
    const char *one1 = p.r_one ? ", one piece each" : "", *one2 = p.c_one ? ", one piece each" : "";
    int r = snprintf(buf, n,
                     "fcs_rowstream_kernel<%d,%d,%d,%s,%s%s> grid %d, shares of %d places%s + fcs_colstream_kernel<%d,%d,%d,%s,%s%s> "
                     "grid %d, shares of %d places, chunks of %d keys%s%s",
                     p.Dp, nb1, p.k1_waves, bf, ps, fold, p.r_blocks, p.r_seg * p.r_unit, one1, p.Dp, p.c_nb, p.c_waves, bf, ps, fold,
                     p.c_blocks, p.c_seg * p.c_unit, p.c_chunk, one2, p.c_direct ? ", direct" : "");
    if (r < 0) return 0;
    const size_t len = (size_t)r;
    if (!p.c_direct) return len + describe_finalize(a, true, len < n ? buf + len : nullptr, len < n ? n - len : 0);
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
