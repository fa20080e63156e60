"""The batch's schedule search on the shortest recordings (its untimed frames
stay within them), and what it reports: a time of the default schedule, and the
default blocks per CU for schedules of one particle per lane, whose grid is a
block per tile."""
import numpy as np
import pytest

import oracle
from mkfbodytracker_pdaf_amd import synthetic
from mkfbodytracker_pdaf_amd.batch import RbpfBatch
from mkfbodytracker_pdaf_amd.devmem import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 2, 3, 6])
def test_autotune_short(T):
    Ns, Ts, K = [300, 70], [T, max(1, T - 1)], 15
    models = [synthetic.make_model(seed=20 + s, K=K) for s in range(2)]
    seqs = [synthetic.simulate(models[s], Ts[s], seed=30 + s, cand_per_joint=4, cap=8) for s in range(2)]
    bins = [oracle.resample_linear(models[s].weights, Ns[s], 40 + s)[0] for s in range(2)]
    b = RbpfBatch(Ns, Ts, K=K, m=6, cand_capacity=8)
    for s, m in enumerate(models):
        b.load_model(s, m.means, m.covs, m.weights, m.gamma, m.pca_proj, m.pca_mean, m.sel, m.R)
    b.set_joint_clutter(models[0].clutter)
    dev = [DeviceArray(np.concatenate([getattr(q, f) for q in seqs]).astype(t))
           for f, t in (("count", np.int32), ("cand", np.float32), ("uniforms", np.uint32))]
    lml = DeviceArray.empty(sum(Ts), np.float64)

    def reset():
        for s in range(2):
            b.reset(s, bins[s])

    reset()
    b.run_dev(*(d.ptr for d in dev), lml.ptr)
    want = lml.get()
    reset()
    best, best_ms, default_ms = b.autotune(*(d.ptr for d in dev), lml.ptr, frames=16)
    assert 0.0 < best_ms <= default_ms
    assert best[1] == 2 or best[2] == 2
    assert tuple(b.schedule) == tuple(best)
    reset()
    b.run_dev(*(d.ptr for d in dev), lml.ptr)
    assert np.array_equal(lml.get(), want)
    b.close()
