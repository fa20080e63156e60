"""A tracker frame that an arm's kernels refuse: the call reports it and leaves
both arms' tracks as they were, and the frame captured next runs.  A tracker
destroyed after its arms."""
import numpy as np
import pytest

from mkfbodytracker_pdaf_amd import capi, synthetic
from mkfbodytracker_pdaf_amd.devmem import DeviceArray
from mkfbodytracker_pdaf_amd.rbpf import Rbpf
from mkfbodytracker_pdaf_amd.tracker import PoseTracker

pytestmark = pytest.mark.gpu

SEL = np.array([9, 10, 0, 1, 12, 13], np.int32)
N, NPOSE = 300, 22


def _arm(seed, d, degenerate=False):
    """An arm on the tracker's pose vector.  degenerate: two measured joints
    share their rows of H, so the state has no selection basis (which the
    24-dimensional state's kernels need)."""
    rng = np.random.default_rng(seed)
    mdl = synthetic.make_model(seed=seed, K=5, d=d)
    proj = rng.standard_normal((d, NPOSE))
    if degenerate:
        proj[:, SEL[2:4]] = proj[:, SEL[0:2]]
    mean = rng.uniform(100.0, 400.0, NPOSE)
    f = Rbpf(N)
    f.load_model(mdl.means, mdl.covs, mdl.weights, mdl.gamma, proj, mean, sel=SEL)
    f.reset(rng.integers(0, 5, N).astype(np.int32))
    return f, proj, mean


def _state(arms):
    return [v for a in arms for v in a.get_tracks() + (a.estimate(),)]


@pytest.mark.parametrize("refused", [0, 1])
def test_refused_frame_leaves_tracks(refused):
    parts = [_arm(3, 12), _arm(4, 24, degenerate=True)]
    if refused == 0:
        parts.reverse()
    arms = [p[0] for p in parts]
    tr = PoseTracker(arms[0], arms[1], parts[0][1], parts[0][2], parts[1][1], parts[1][2], seed=2)
    imgs, rois = synthetic.tracker_sequence(2, seed=8)
    before = _state(arms)
    with pytest.raises(capi.PfError):
        tr.callback(imgs[0], rois[0])
    assert all(np.array_equal(p, q) for p, q in zip(_state(arms), before))
    dev = DeviceArray(imgs), DeviceArray(rois)
    with pytest.raises(capi.PfError):
        tr.run_dev(2, dev[0].ptr, dev[1].ptr)
    tr.synchronize()
    assert all(np.array_equal(p, q) for p, q in zip(_state(arms), before))
    # the arm gets a model that its kernels take: the frame runs
    good, proj, mean = _arm(5, 24)
    mdl = synthetic.make_model(seed=5, K=5, d=24)
    arms[refused].load_model(mdl.means, mdl.covs, mdl.weights, mdl.gamma, proj, mean, sel=SEL)
    arms[refused].reset(np.zeros(N, np.int32))
    out = tr.callback(imgs[0], rois[0])
    assert np.all(np.isfinite(out["lml"])) and np.all(np.isfinite(out["pose"]))
    assert not np.array_equal(_state(arms)[0], before[0])
    tr.close()
    for a in arms + [good]:
        a.close()


@pytest.mark.parametrize("d2", [12, 16])     # the arms in paired launches, and on a stream each
def test_tracker_destroyed_after_its_arms(d2):
    parts = [_arm(3, 12), _arm(4, d2)]
    arms = [p[0] for p in parts]
    tr = PoseTracker(arms[0], arms[1], parts[0][1], parts[0][2], parts[1][1], parts[1][2], seed=2)
    imgs, rois = synthetic.tracker_sequence(2, seed=8)
    dev = DeviceArray(imgs), DeviceArray(rois)
    tr.callback(imgs[0], rois[0])
    tr.run_dev(2, dev[0].ptr, dev[1].ptr)    # captured frames of both kinds, the last run not waited for
    for a in arms:
        a.close()
    tr.close()
