// wr_many_mixed.hip -- the one-launch band kernel of small tiles (mixed precision, McICA route).
#include "wr_many.h"

namespace wr {
template int launch_many<float, false, false>(const BandJob<float> &, hipStream_t);
}  // namespace wr
