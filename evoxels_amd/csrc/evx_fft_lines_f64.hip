// Runtime-radix line transforms, float64.
#include "evx_fft_line_kernels.hpp"

namespace evx {
EVX_LINE_INSTANTIATE(double)
}  // namespace evx
