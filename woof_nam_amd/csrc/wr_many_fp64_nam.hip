// wr_many_fp64_nam.hip -- the optics and sweep kernels of small tiles (FP64, NAM route; wr_many.h).
#include "wr_many.h"

namespace wr {
template int launch_many<double, true, false>(const BandJob<double> &, hipStream_t);
}  // namespace wr
