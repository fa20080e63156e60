"""Models loaded again into a batch that already ran (one sequence, every
sequence, and under another joint order): the next run equals that of a new
batch loaded once with the same models, bit for bit."""
import numpy as np
import pytest

import oracle
from mkfbodytracker_pdaf_amd import synthetic
from mkfbodytracker_pdaf_amd.batch import RbpfBatch
from mkfbodytracker_pdaf_amd.devmem import DeviceArray

pytestmark = pytest.mark.gpu

NS, TS, CAP = [300, 1, 513], [3, 5, 4], 8


def _load(b, which, models):
    for s in which:
        m = models[s]
        b.load_model(s, m.means, m.covs, m.weights, m.gamma, m.pca_proj, m.pca_mean, m.sel, m.R)


def _run(b, models, clutter, inputs):
    b.set_joint_clutter(clutter)
    for s, n in enumerate(NS):
        b.reset(s, oracle.resample_linear(models[s].weights, n, 77 + s)[0])
    cnt, cand, uni, lml = inputs
    b.run_dev(cnt.ptr, cand.ptr, uni.ptr, lml.ptr)
    return lml.get(), [b.get_tracks(s) for s in range(len(NS))], [b.estimate(s) for s in range(len(NS))]


@pytest.mark.parametrize("again", [[1], [0, 1, 2], []])
@pytest.mark.parametrize("clutter", [[0, 1, 1], [1, 0, 1]])
def test_reloaded_batch_equals_new_batch(again, clutter):
    first = [synthetic.make_model(seed=3 + s) for s in range(3)]
    second = [synthetic.make_model(seed=30 + s) if s in again else first[s] for s in range(3)]
    seqs = [synthetic.simulate(second[s], t, seed=50 + s, cap=CAP) for s, t in enumerate(TS)]
    inputs = [DeviceArray(np.concatenate([q.count for q in seqs]).astype(np.int32)),
              DeviceArray(np.concatenate([q.cand for q in seqs]).astype(np.float32)),
              DeviceArray(np.concatenate([q.uniforms for q in seqs]).astype(np.uint32)),
              DeviceArray.empty(sum(TS), np.float64)]
    old, new = (RbpfBatch(NS, TS, K=first[0].K, m=first[0].m, cand_capacity=CAP) for _ in range(2))
    _load(old, range(3), first)
    _run(old, first, [0, 1, 1], inputs)
    _load(old, again, second)
    got = _run(old, second, clutter, inputs)
    _load(new, range(3), second)
    want = _run(new, second, clutter, inputs)
    assert np.array_equal(got[0], want[0])
    for s in range(3):
        assert all(np.array_equal(a, b) for a, b in zip(got[1][s], want[1][s]))
        assert np.array_equal(got[2][s], want[2][s])
    old.close()
    new.close()
