// FP64 full-spectrum transforms of real input.
#include "jt_real1d.hpp"

namespace jt {
JT_FULL_INST(, double)
}  // namespace jt
