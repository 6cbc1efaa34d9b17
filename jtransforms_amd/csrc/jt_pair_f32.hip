// FP32 real transforms that run two lines as one complex transform.
#include "jt_pair.hpp"

namespace jt {
JT_PAIR_INST(, float)
}  // namespace jt
