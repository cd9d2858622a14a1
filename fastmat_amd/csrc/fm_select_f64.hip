// Selected-element passes of complex128 (see fm_select_launch.hpp).
#include "fm_select_launch.hpp"

namespace fm {
template fm_status launch_select<double>(const TileArgs<double> &, const SelectArgs<double> &, hipStream_t);
}  // namespace fm
