// wr_many_mixed_nam.hip -- the one-launch band kernel of small tiles (mixed precision, NAM route).
#include "wr_many.h"

namespace wr {
template int launch_many<float, true, false>(const BandJob<float> &, hipStream_t);
}  // namespace wr
