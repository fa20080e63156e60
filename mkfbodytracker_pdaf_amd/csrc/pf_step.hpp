// pf_step.hpp -- launches of the single-filter step (k_step), one source per
// state layout (pf_step_rec.hip, pf_step_rows.hip), so that their many kernels
// compile side by side.
#pragma once

#include "pf_kernels.hpp"

namespace mkfbt {

struct StepLaunch {
    int D, J, N, block, mode;     // state dimension, joints, particles, threads per block, StepMode
    bool sel;                     // selection basis
    hipStream_t stream;
};

int launch_step_rec(const StepLaunch &s, const StepArgs &a);     // per-particle records (d <= 12)
int launch_step_rows(const StepLaunch &s, const StepArgs &a);    // rows

template <int D, int SELJ, bool REC>
int launch_step_dj(const StepLaunch &s, const StepArgs &a)
{
    const size_t lds = (size_t)step_lds_bytes_rec(REC, a.stage_floats, a.anc_mode == kAncFused ? a.pend.nb : 0);
    // fused launches have one more block, for the frame's statistics
    const int grid = (s.N + s.block - 1) / s.block + (a.anc_mode == kAncFused ? 1 : 0);
    if (s.mode == kModeRef)
        hipLaunchKernelGGL((k_step<D, kModeRef, SELJ, REC>), dim3(grid), dim3(s.block), lds, s.stream, a);
    else
        hipLaunchKernelGGL((k_step<D, kModeCand, SELJ, REC>), dim3(grid), dim3(s.block), lds, s.stream, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(PF_ERR_HIP, "k_step launch failed: %s", hipGetErrorString(e));
    return PF_OK;
}

// Selection-basis kernels exist for every joint count J with 2J <= D.
template <int D, bool REC>
int launch_step_d(const StepLaunch &s, const StepArgs &a)
{
    if (!s.sel) return launch_step_dj<D, 0, REC>(s, a);
    switch (s.J) {
    case 1: return launch_step_dj<D, 1, REC>(s, a);
    case 2: return launch_step_dj<D, 2, REC>(s, a);
    case 3: return launch_step_dj<D, 3, REC>(s, a);
    case 4: return launch_step_dj<D, 4, REC>(s, a);
    case 5: if constexpr (D >= 10) return launch_step_dj<D, 5, REC>(s, a); break;
    case 6: if constexpr (D >= 12) return launch_step_dj<D, 6, REC>(s, a); break;
    case 7: if constexpr (D >= 14) return launch_step_dj<D, 7, REC>(s, a); break;
    case 8: if constexpr (D >= 16) return launch_step_dj<D, 8, REC>(s, a); break;
    default: break;
    }
    return launch_step_dj<D, 0, REC>(s, a);
}

}  // namespace mkfbt
