// Shrinkage passes of complex64 (see fm_shrink_launch.hpp).
#include "fm_shrink_launch.hpp"

namespace fm {
template fm_status launch_shrink<float, false>(const TileArgs<float> &, const ShrinkArgs<float> &,
                                          hipStream_t);
template fm_status launch_shrink<float, true>(const TileArgs<float> &, const ShrinkArgs<float> &,
                                         hipStream_t);
}  // namespace fm
