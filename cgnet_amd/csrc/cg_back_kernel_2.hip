#include "cg_back_kernel.h"

namespace cgnet {
CGNET_BACK_VARIANT(2, 4, 2)
}  // namespace cgnet
