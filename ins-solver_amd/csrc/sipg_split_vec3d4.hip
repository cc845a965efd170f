// Four-wave element passes of the vector (velocity) operator with slip faces (sipg_split.h), 3D order 4.
#include "sipg_split_kernels.h"

namespace insp {
namespace split {
INSP_SPLIT_VEC(, 3, 4)
}  // namespace split
}  // namespace insp
