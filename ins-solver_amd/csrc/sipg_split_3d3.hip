// Four-wave trace and element passes of 3D order 3 (sipg_split.h).
#include "sipg_split_kernels.h"

namespace insp {
namespace split {
INSP_SPLIT_INST(, 3, 3, double)
INSP_SPLIT_INST(, 3, 3, float)
}  // namespace split
}  // namespace insp
