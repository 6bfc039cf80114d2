#include "cg_back_kernel.h"

namespace cgnet {
CGNET_BACK_VARIANT(3, 4, 3)
}  // namespace cgnet
