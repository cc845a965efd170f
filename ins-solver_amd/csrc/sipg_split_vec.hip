// Four-wave element passes of the vector (velocity) operator with slip faces (sipg_split.h).
#include "sipg_split_kernels.h"

namespace insp {
namespace split {
INSP_SPLIT_VEC(, 2, 2)
INSP_SPLIT_VEC(, 2, 3)
INSP_SPLIT_VEC(, 2, 4)
INSP_SPLIT_VEC(, 3, 2)
INSP_SPLIT_VEC(, 3, 3)
}  // namespace split
}  // namespace insp
