// Instantiation unit of segmented.hpp.
#include "segmented.hpp"

namespace bcmi {

BCMI_SEGPLAN_SIGNATURE(segplan_run_u32) { return run_plan_vb<uint32_t>(q, pl, keys, vals); }

}  // namespace bcmi
