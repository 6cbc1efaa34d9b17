// FP64 DCT, DST and DHT.
#include "jt_r2r.hpp"

namespace jt {
JT_R2R_INST(, double)
}  // namespace jt
