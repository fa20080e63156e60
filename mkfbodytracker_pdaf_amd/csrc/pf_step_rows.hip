// pf_step_rows.hip -- the single-filter step on rows (structure of arrays).
#include <hip/hip_runtime.h>

#include "../../include/pf_rbpf.h"
#include "pf_internal.hpp"
#include "pf_step.hpp"

namespace mkfbt {

int launch_step_rows(const StepLaunch &s, const StepArgs &a)
{
    switch (s.D) {
    case 8: return launch_step_d<8, false>(s, a);
    case 12: return launch_step_d<12, false>(s, a);
    case 16: return launch_step_d<16, false>(s, a);
    case 24:
        // compiled for 3 and 5 joints in the selection basis (the
        // scaled-state workloads); other joint counts report unsupported
        if (s.sel && s.J == 3) return launch_step_dj<24, 3, false>(s, a);
        if (s.sel && s.J == 5) return launch_step_dj<24, 5, false>(s, a);
        return set_error(PF_ERR_UNSUPPORTED, "d = 24 is compiled for 3 or 5 joints with a full-rank H");
    default: return set_error(PF_ERR_UNSUPPORTED, "state dimension %d not compiled", s.D);
    }
}

}  // namespace mkfbt
