// Selected-element passes of complex64 (see fm_select_launch.hpp).
#include "fm_select_launch.hpp"

namespace fm {
template fm_status launch_select<float>(const TileArgs<float> &, const SelectArgs<float> &, hipStream_t);
}  // namespace fm
