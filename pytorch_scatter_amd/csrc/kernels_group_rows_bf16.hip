// Kernel instantiations of the group statistics over sorted entries for element type bf16_t.
#include "group_rows.h"

namespace ts {
TS_INSTANTIATE_GROUP_ROWS(bf16_t)
}  // namespace ts
