// Shrinkage passes of complex128 (see fm_shrink_launch.hpp).
#include "fm_shrink_launch.hpp"

namespace fm {
template fm_status launch_shrink<double, false>(const TileArgs<double> &, const ShrinkArgs<double> &,
                                          hipStream_t);
template fm_status launch_shrink<double, true>(const TileArgs<double> &, const ShrinkArgs<double> &,
                                         hipStream_t);
}  // namespace fm
