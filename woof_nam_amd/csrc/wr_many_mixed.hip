// wr_many_mixed.hip -- the optics and sweep kernels of small tiles (mixed precision, McICA route; wr_many.h).
#include "wr_many.h"

namespace wr {
template int launch_many<float, false, false>(const BandJob<float> &, hipStream_t);
}  // namespace wr
