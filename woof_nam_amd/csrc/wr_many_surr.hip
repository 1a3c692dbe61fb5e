// wr_many_surr.hip -- the two launches of small tiles (mixed precision, learned gas optics, McICA route).
#include "wr_many.h"

namespace wr {
template int launch_many<float, false, true>(const BandJob<float> &, hipStream_t);
}  // namespace wr
