// Plain pass kernels of complex128 (see fm_fft_launch.hpp).
#include "fm_fft_launch.hpp"

namespace fm {
template fm_status launch_kind<double, false>(const TileArgs<double> &, hipStream_t);
}  // namespace fm
