// FP32 full-spectrum transforms of real input.
#include "jt_real1d.hpp"

namespace jt {
JT_FULL_INST(, float)
}  // namespace jt
