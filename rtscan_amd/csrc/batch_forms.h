// batch_forms.h -- for the autotuner: a plan without queries that are evaluated together.
#pragma once

#include "rts_batch.h"

namespace rts {

// Whether the queries that are planned from now on (rts_batch_plan_set_queries, _set_config) are
// all evaluated by their columns' forms.
void batch_plan_all_apart(rts_batch_plan *plan, bool apart);

}  // namespace rts
