// The complex engine's FP64 forward transforms.
#include "jt_fft1d.hpp"

namespace jt {
JT_C2C_INST(, double, -1)
}  // namespace jt
