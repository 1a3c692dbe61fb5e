// wr_many_mixed_nam.hip -- the optics and sweep kernels of small tiles (mixed precision, NAM route; wr_many.h).
#include "wr_many.h"

namespace wr {
template int launch_many<float, true, false>(const BandJob<float> &, hipStream_t);
}  // namespace wr
