// Kernel instantiations of the group statistics over sorted entries for element type double.
#include "group_rows.h"

namespace ts {
TS_INSTANTIATE_GROUP_ROWS(double)
}  // namespace ts
