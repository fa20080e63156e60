"""The d = 24 batch's two state layouts (a record per particle for the four-lane
kernels, rows for the kernel of one particle per lane), around their tiles'
and waves' edges: the same initial tracks bit for bit, imported tracks back to FP32
rounding, the state carried over a change of kernel, and equal runs whether the
kernel was chosen before or after the reset."""
import numpy as np
import pytest

import oracle
from mkfbodytracker_pdaf_amd import capi, synthetic
from mkfbodytracker_pdaf_amd.batch import RbpfBatch
from mkfbodytracker_pdaf_amd.devmem import DeviceArray

pytestmark = pytest.mark.gpu

ROWS, QUAD, MFMA = capi.PF_BATCH_VALU, capi.PF_BATCH_QUAD_VALU, capi.PF_BATCH_MFMA
NS, T = [1, 15, 17, 255, 257, 600], 2


def _setup(K, joints):
    J = len(joints)
    models = [synthetic.make_model(seed=7 + s, K=K, d=24, joints=joints, clutter=(1,) * J) for s in range(len(NS))]
    seqs = [synthetic.simulate(models[s], T, seed=30 + s, cand_per_joint=5, cap=16) for s in range(len(NS))]
    bins = [oracle.resample_linear(models[s].weights, NS[s], 40 + s)[0] for s in range(len(NS))]
    b = RbpfBatch(NS, [T] * len(NS), K=K, m=2 * J, d=24, cand_capacity=16)
    for s, m in enumerate(models):
        b.load_model(s, m.means, m.covs, m.weights, m.gamma, m.pca_proj, m.pca_mean, m.sel, m.R)
    b.set_joint_clutter(models[0].clutter)
    dev = [DeviceArray(np.concatenate([getattr(q, f) for q in seqs]).astype(t))
           for f, t in (("count", np.int32), ("cand", np.float32), ("uniforms", np.uint32))]
    return b, bins, dev


def _state(b):
    return [b.get_tracks(s) + (b.estimate(s),) for s in range(len(NS))]


def _equal(p, q):
    return all(np.array_equal(a, c) for u, v in zip(p, q) for a, c in zip(u, v))


@pytest.mark.parametrize("K,joints", [
    (64, ("head", "left_hand", "right_hand", "left_elbow", "right_elbow")),
    (15, ("head", "left_hand", "right_hand"))])
def test_layouts(K, joints):
    b, bins, dev = _setup(K, joints)
    lml = DeviceArray.empty(T * len(NS), np.float64)

    def reset(variant):
        b.variant = variant
        for s, bi in enumerate(bins):
            b.reset(s, bi)

    def run():
        b.run_dev(*(d.ptr for d in dev), lml.ptr)
        return _state(b), lml.get()

    # initial tracks (T is even, so buffer 0 is the one read)
    reset(ROWS)
    first = _state(b)
    b.variant = MFMA                       # carried into records ...
    assert _equal(_state(b), first)
    b.variant = ROWS                       # ... and back
    assert _equal(_state(b), first)
    want_rows = run()
    reset(MFMA)
    assert _equal(_state(b), first)
    # imported tracks: to FP32 rounding of T x and T P T^T (condition of the basis below 1e3)
    for s in range(len(NS)):
        b.set_tracks(s, first[s][0], first[s][1])
    for u, v in zip(_state(b), first):
        for a, c in zip(u, v):
            assert np.abs(a - c).max() <= 1e-3 * np.abs(c).max()
    # the kernel chosen before and after the reset
    for variant in (MFMA, QUAD):
        reset(variant)
        want = run()
        after = _state(b)
        b.variant = ROWS                   # a run's final state, carried over
        assert _equal(_state(b), after)
        reset(ROWS)
        b.variant = variant
        got = run()
        assert _equal(got[0], want[0]) and np.array_equal(got[1], want[1])
    reset(MFMA)
    b.variant = ROWS
    got = run()
    assert _equal(got[0], want_rows[0]) and np.array_equal(got[1], want_rows[1])
    b.close()
