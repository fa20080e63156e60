"""Model images around the sizes where the step's LDS (the staged image, then
the record gather's slices) passes 64 KB, half a CU's and the budget above
which the component rows stay in global memory: a device-resident run equals
host-driven steps bit for bit in both state layouts, and the component draw
equals the oracle's."""
import numpy as np
import pytest

import oracle
from mkfbodytracker_pdaf_amd import capi, synthetic
from mkfbodytracker_pdaf_amd.devmem import DeviceArray
from mkfbodytracker_pdaf_amd.rbpf import Rbpf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1, 2, 43, 47, 90, 110, 126, 140])
@pytest.mark.parametrize("N", [33, 700])
def test_run_equals_host_steps(K, N):
    T, cap = 4, 8
    mdl = synthetic.make_model(seed=K, K=K)
    seq = synthetic.simulate(mdl, T, seed=K + 1, cand_per_joint=4, cap=cap)
    bins = oracle.resample_linear(mdl.weights, N, 3)[0]
    dev = [DeviceArray(a) for a in (seq.count.astype(np.int32), seq.cand.astype(np.float32),
                                    seq.uniforms.astype(np.uint32))]
    d_lml = DeviceArray.empty(T, np.float64)
    seen = []
    for layout in (capi.PF_LAYOUT_ROWS, capi.PF_LAYOUT_RECORDS):
        rb = Rbpf(N, cand_capacity=cap)
        rb.load_model(mdl.means, mdl.covs, mdl.weights, mdl.gamma, mdl.pca_proj, mdl.pca_mean, sel=mdl.sel, R=mdl.R)
        rb.set_joint_clutter(mdl.clutter)
        rb.state_layout = layout
        rb.reset(bins)
        want = []
        for t in range(T):
            u = [int(v) for v in seq.uniforms[t]]
            out = rb.step_candidates(seq.count[t], seq.cand[t], *u)[1]
            want.append(out["lml"])
            assert np.array_equal(out["comp"], oracle.resample_linear(mdl.weights, N, u[0])[0])
        tracks = rb.get_tracks()
        for flags in (0, 1):
            rb.reset(bins)
            rb.run_candidates_dev(T, dev[0].ptr, dev[1].ptr, dev[2].ptr, d_lml.ptr, flags)
            assert rb.synchronize() == 0
            assert np.array_equal(d_lml.get(), np.array(want))
            assert all(np.array_equal(a, b) for a, b in zip(rb.get_tracks(), tracks))
        seen.append((want, tracks))
        rb.close()
    assert seen[0][0] == seen[1][0]
    assert all(np.array_equal(a, b) for a, b in zip(seen[0][1], seen[1][1]))
