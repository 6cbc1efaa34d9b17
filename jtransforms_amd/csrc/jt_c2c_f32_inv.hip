// The complex engine's FP32 backward transforms.
#include "jt_fft1d.hpp"

namespace jt {
JT_C2C_INST(, float, 1)
}  // namespace jt
