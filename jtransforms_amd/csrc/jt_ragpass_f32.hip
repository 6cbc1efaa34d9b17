// FP32 ragged batches, one launch per pass.
#include "jt_ragpass.hpp"

namespace jt {
JT_RAGPASS_INST(, float)
}  // namespace jt
