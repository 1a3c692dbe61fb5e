// wr_many_fp64.hip -- the optics and sweep kernels of small tiles (FP64, McICA route; wr_many.h).
#include "wr_many.h"

namespace wr {
template int launch_many<double, false, false>(const BandJob<double> &, hipStream_t);
}  // namespace wr
