"""Component counts of the d = 24 batch around those whose image would fill the
LDS budget together with the resampler's workspace (30 to 36 here).  The
four-lane kernels stage the image without its component rows and take all of
them: one frame against the oracle.  The kernel of one particle per lane stages
the rows too and refuses those."""
import numpy as np
import pytest

import oracle
from mkfbodytracker_pdaf_amd import capi, synthetic
from mkfbodytracker_pdaf_amd.batch import RbpfBatch
from mkfbodytracker_pdaf_amd.devmem import DeviceArray

pytestmark = pytest.mark.gpu

JOINTS = ("head", "left_hand", "right_hand", "left_elbow", "right_elbow")
N, CAP, LAM, GATE = 600, 16, 4 / (640.0 * 480.0), 9.210340371976184


def _batch(K):
    mdl = synthetic.make_model(seed=K, K=K, d=24, joints=JOINTS, clutter=(1,) * 5)
    seq = synthetic.simulate(mdl, 1, seed=K + 1, cand_per_joint=5, cap=CAP)
    b = RbpfBatch([N], [1], K=K, m=10, d=24, cand_capacity=CAP, clutter_density=LAM)
    b.load_model(0, mdl.means, mdl.covs, mdl.weights, mdl.gamma, mdl.pca_proj, mdl.pca_mean, mdl.sel, mdl.R)
    b.set_joint_clutter(mdl.clutter)
    dev = [DeviceArray(a) for a in (seq.count.astype(np.int32), seq.cand.astype(np.float32),
                                    seq.uniforms.astype(np.uint32))] + [DeviceArray.empty(1, np.float64)]
    return b, mdl, seq, dev


@pytest.mark.parametrize("variant", [capi.PF_BATCH_MFMA, capi.PF_BATCH_QUAD_VALU])
@pytest.mark.parametrize("K", [28, 29, 32, 36, 37])
def test_four_lane_kernels(variant, K):
    b, mdl, seq, dev = _batch(K)
    b.variant = variant
    bins = oracle.resample_linear(mdl.weights, N, 3)[0]
    b.reset(0, bins)
    b.run_dev(*(d.ptr for d in dev))
    om = oracle.Model(mdl.weights, mdl.gamma, mdl.means, mdl.Sigma, mdl.H(), mdl.BH(), mdl.R)
    U1, U2 = (int(u) for u in seq.uniforms[0])
    ref = om.update_pdaf(*om.reset(bins), mdl.clutter, seq.count[0], seq.cand[0], U1, U2, 0.95, GATE, LAM)
    # FP32 state and likelihoods against FP64 (the bound of the d = 24 tests)
    lw, anc = b.last_frame(0)
    assert np.all(np.abs(lw - ref["lw"]) <= 1e-4 * np.maximum(1.0, np.abs(ref["lw"])))
    assert np.array_equal(anc, oracle.resample_log(lw.astype(np.float64), N, U2)[0])
    x, P = b.get_tracks(0)
    for got, want in ((x, ref["xu"][anc]), (P, ref["Pu"][anc])):
        got, want = got.reshape(N, -1), want.reshape(N, -1)
        assert np.all(np.linalg.norm(got - want, axis=1) <= 1e-4 * np.linalg.norm(want, axis=1))
    b.close()


@pytest.mark.parametrize("K,refused", [(28, False), (32, True), (36, True), (37, False)])
def test_one_particle_per_lane(K, refused):
    b, mdl, _, dev = _batch(K)
    b.variant = capi.PF_BATCH_VALU
    b.reset(0, oracle.resample_linear(mdl.weights, N, 3)[0])
    if refused:
        with pytest.raises(capi.PfError):
            b.run_dev(*(d.ptr for d in dev))
    else:
        assert b.run_dev(*(d.ptr for d in dev)) == 0
    b.close()
