// Shrinkage passes of complex128 (see fm_shrink_launch.hpp).
#include "fm_shrink_launch.hpp"

namespace fm {
#define FM_PASS(P) \
    template fm_status launch_shrink<double, P>(const TileArgs<double> &, const ShrinkArgs<double> &, \
                                               hipStream_t);
FM_PASS(SHRINK_COLUMN)
FM_PASS(SHRINK_CONV)
FM_PASS(SHRINK_NEXT)
}  // namespace fm
