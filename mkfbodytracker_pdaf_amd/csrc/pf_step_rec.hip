// pf_step_rec.hip -- the single-filter step on per-particle records.
#include <hip/hip_runtime.h>

#include "../../include/pf_rbpf.h"
#include "pf_internal.hpp"
#include "pf_step.hpp"

namespace mkfbt {

int launch_step_rec(const StepLaunch &s, const StepArgs &a)
{
    switch (s.D) {
    case 8: return launch_step_d<8, true>(s, a);
    case 12: return launch_step_d<12, true>(s, a);
    default: return set_error(PF_ERR_UNSUPPORTED, "records are compiled for d <= 12");
    }
}

}  // namespace mkfbt
