// Four-wave trace and element passes of 3D order 4, FP64 (sipg_split.h).
#include "sipg_split_kernels.h"

namespace insp {
namespace split {
INSP_SPLIT_INST(, 3, 4, double)
}  // namespace split
}  // namespace insp
