// Kernel instantiations of the group statistics over sorted entries for element type f16_t.
#include "group_rows.h"

namespace ts {
TS_INSTANTIATE_GROUP_ROWS(f16_t)
}  // namespace ts
