// wr_many_fp64.hip -- the one-launch band kernel of small tiles (FP64, McICA route).
#include "wr_many.h"

namespace wr {
template int launch_many<double, false, false>(const BandJob<double> &, hipStream_t);
}  // namespace wr
