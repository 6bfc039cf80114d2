#include "cg_back_kernel.h"

namespace cgnet {
CGNET_BACK_VARIANT(0, 2, 1)
}  // namespace cgnet
