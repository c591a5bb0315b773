// Column pass of the two-pass path, the rows of a key head's query heads laid end to end.
#include "fcs_stream_kernels.h"

namespace fcs {

template hipError_t launch_colstream_f<true>(const Plan &, const Args &, hipStream_t);

}  // namespace fcs
