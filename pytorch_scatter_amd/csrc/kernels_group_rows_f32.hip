// Kernel instantiations of the group statistics over sorted entries for element type float.
#include "group_rows.h"

namespace ts {
TS_INSTANTIATE_GROUP_ROWS(float)
}  // namespace ts
