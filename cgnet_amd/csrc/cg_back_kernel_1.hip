#include "cg_back_kernel.h"

namespace cgnet {
CGNET_BACK_VARIANT(1, 3, 2)
}  // namespace cgnet
