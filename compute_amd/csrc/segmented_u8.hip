// Instantiation unit of segmented.hpp.
#include "segmented.hpp"

namespace bcmi {

BCMI_SEGPLAN_SIGNATURE(segplan_run_u8) { return run_plan_vb<uint8_t>(q, pl, keys, vals); }

}  // namespace bcmi
