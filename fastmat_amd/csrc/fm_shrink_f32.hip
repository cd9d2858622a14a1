// Shrinkage passes of complex64 (see fm_shrink_launch.hpp).
#include "fm_shrink_launch.hpp"

namespace fm {
#define FM_PASS(P) \
    template fm_status launch_shrink<float, P>(const TileArgs<float> &, const ShrinkArgs<float> &, \
                                               hipStream_t);
FM_PASS(SHRINK_COLUMN)
FM_PASS(SHRINK_CONV)
FM_PASS(SHRINK_NEXT)
}  // namespace fm
