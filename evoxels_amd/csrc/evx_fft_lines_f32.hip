// Runtime-radix line transforms, float32.
#include "evx_fft_line_kernels.hpp"

namespace evx {
EVX_LINE_INSTANTIATE(float)
}  // namespace evx
