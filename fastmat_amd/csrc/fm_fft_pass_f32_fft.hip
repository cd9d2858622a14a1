// Plain pass kernels of complex64 (see fm_fft_launch.hpp).
#include "fm_fft_launch.hpp"

namespace fm {
template fm_status launch_kind<float, false>(const TileArgs<float> &, hipStream_t);
}  // namespace fm
