// Row-statistics pass of the two-pass path.
#include "fcs_stream_kernels.h"

namespace fcs {

template hipError_t launch_rowstream_f<false>(const Plan &, const Args &, hipStream_t);

}  // namespace fcs
