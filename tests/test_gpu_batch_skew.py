"""A batch of a long recording beside many short ones: the frames after the
short ones' ends launch blocks for the active tiles only, also where captured
frames are replayed (a pair captured again after the ends of frames 2 and 201,
between an odd and an even frame too).  Every sequence's log mean weights equal
those of launches one by one and of other tile sizes bit for bit."""
import numpy as np
import pytest

import oracle
from mkfbodytracker_pdaf_amd import synthetic
from mkfbodytracker_pdaf_amd.batch import RbpfBatch
from mkfbodytracker_pdaf_amd.devmem import DeviceArray

pytestmark = pytest.mark.gpu

CASES = {12: ([300] + [20000] * 60, [1000] + [201] * 40 + [2] * 20, 3, ((64, 1, 2), (128, 1, 2), (256, 1, 2), (256, 2, 2))),
         24: ([300] + [9000] * 60, [2001] + [2] * 60, 3, ((256, 1, 2),))}


@pytest.mark.parametrize("d", [12, 24])
def test_skewed_lengths(d):
    Ns, Ts, J, schedules = CASES[d]
    S, K = len(Ns), 5
    models = [synthetic.make_model(seed=20 + s % 3, K=K, d=d) for s in range(S)]
    seqs = [synthetic.simulate_fast(models[s], Ts[s], seed=30 + s, cand_per_joint=4, cap=8) for s in range(S)]
    bins = [oracle.resample_linear(models[s].weights, Ns[s], 40 + s)[0] for s in range(S)]
    b = RbpfBatch(Ns, Ts, K=K, m=2 * J, d=d, cand_capacity=8)
    for s, m in enumerate(models):
        b.load_model(s, m.means, m.covs, m.weights, m.gamma, m.pca_proj, m.pca_mean, m.sel, m.R)
    b.set_joint_clutter(models[0].clutter)
    dev = [DeviceArray(np.concatenate([getattr(q, f) for q in seqs]).astype(t))
           for f, t in (("count", np.int32), ("cand", np.float32), ("uniforms", np.uint32))]
    lml = DeviceArray.empty(sum(Ts), np.float64)
    want = None
    for schedule in schedules:
        b.schedule = schedule
        for graph in (False, True):
            for s, bi in enumerate(bins):
                b.reset(s, bi)
            b.run_dev(*(a.ptr for a in dev), lml.ptr, graph=graph)
            got = lml.get(), [b.estimate(s) for s in (0, 1, S - 1)]
            want = got if want is None else want
            assert np.array_equal(got[0], want[0]), (schedule, graph)
            assert all(np.array_equal(p, q) for p, q in zip(got[1], want[1])), (schedule, graph)
    assert np.all(np.isfinite(want[0]))
    b.close()
