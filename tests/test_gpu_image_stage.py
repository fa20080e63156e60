"""Model images around the size beside which the record rounds' LDS leaves two
blocks per CU (up to K = 90 for this shape; above, the component rows stay in global
memory in records and are staged in rows): runs over more blocks than CUs equal in
both layouts bit for bit, also when the layout changes with tracks in place."""
import numpy as np
import pytest

import oracle
from mkfbodytracker_pdaf_amd import capi, synthetic
from mkfbodytracker_pdaf_amd.devmem import DeviceArray
from mkfbodytracker_pdaf_amd.rbpf import Rbpf

pytestmark = pytest.mark.gpu

ROWS, RECORDS = capi.PF_LAYOUT_ROWS, capi.PF_LAYOUT_RECORDS


@pytest.mark.parametrize("K", [90, 91, 92, 126])
@pytest.mark.parametrize("N", [700, 66000])
def test_layouts_equal(K, N):
    T, cap = 2, 8
    mdl = synthetic.make_model(seed=K, K=K)
    seq = synthetic.simulate(mdl, T, seed=K + 1, cand_per_joint=4, cap=cap)
    bins = oracle.resample_linear(mdl.weights, N, 3)[0]
    dev = [DeviceArray(a) for a in (seq.count.astype(np.int32), seq.cand.astype(np.float32),
                                    seq.uniforms.astype(np.uint32))]
    d_lml = DeviceArray.empty(T, np.float64)
    rb = Rbpf(N, cand_capacity=cap)
    rb.load_model(mdl.means, mdl.covs, mdl.weights, mdl.gamma, mdl.pca_proj, mdl.pca_mean, sel=mdl.sel, R=mdl.R)
    rb.set_joint_clutter(mdl.clutter)

    def run():
        rb.run_candidates_dev(T, dev[0].ptr, dev[1].ptr, dev[2].ptr, d_lml.ptr, 1)
        assert rb.synchronize() == 0
        return d_lml.get()

    seen = []
    for first, second in ((ROWS, ROWS), (RECORDS, RECORDS), (RECORDS, ROWS), (ROWS, RECORDS)):
        rb.state_layout = first
        rb.reset(bins)
        lml = [run()]
        rb.state_layout = second
        lml.append(run())
        seen.append((np.concatenate(lml), rb.estimate()))
    for got in seen[1:]:
        assert all(np.array_equal(a, b) for a, b in zip(got, seen[0]))
    rb.close()
