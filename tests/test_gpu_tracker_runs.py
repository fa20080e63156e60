"""Device-resident tracker runs replayed from captured groups of frames: every
output equals the frames launched one by one, over run lengths around the group
sizes, on one tracker used for several runs, after its arms' state buffers
changed roles (odd lengths), were reset, and had their resampler scratch and
model tables allocated again, and after a longer run grew its buffers."""
import os

import numpy as np
import pytest

from mkfbodytracker_pdaf_amd import synthetic
from mkfbodytracker_pdaf_amd.devmem import DeviceArray
from mkfbodytracker_pdaf_amd.tracker import PoseTracker

pytestmark = pytest.mark.gpu

ARMS = [os.path.join(os.path.dirname(__file__), "golden", f"data{a}_PCA_100000_15_12.yml") for a in ("13D", "23D")]


def _run(tr, T, dev, graph):
    out = [DeviceArray.empty(s, np.float64) for s in ((2, T), (T, 2, 22), (T, 2, 15), (T, 24), (T, 16))]
    tr.run_dev(T, dev[0].ptr, dev[1].ptr, *(o.ptr for o in out), graph=graph)
    tr.synchronize()
    last = tr.get_last()
    return [o.get() for o in out] + [last["blurred"], last["bins"], last["Z"]]


@pytest.mark.parametrize("N", [100, 513])
def test_replayed_groups_equal_launched_frames(N):
    imgs, rois = synthetic.tracker_sequence(70, seed=4)
    dev = DeviceArray(imgs), DeviceArray(rois)
    pair = [PoseTracker.from_yml(*ARMS, n_particles=N, seed=9) for _ in range(2)]
    for step, T in enumerate((1, 2, 17, 15, 33, 16, 70, 31)):
        got, want = (_run(tr, T, dev, graph) for tr, graph in zip(pair, (True, False)))
        for a, b in zip(got, want):
            assert np.array_equal(a, b), (T, step)
        for tr in pair:
            if step == 2:
                for a, arm in enumerate(tr.arms):
                    arm.reset(np.full(N, a, np.int32))
            if step == 3:                     # larger than the proposals' scratch
                tr.arms[1].resample(np.ones(20 * N), 10, 5)
            if step == 5:
                tr.arms[0].set_joint_clutter([0, 0, 0])
    for tr in pair:
        tr.close()


def test_frame_calls_equal_run():
    T, N = 5, 300
    imgs, rois = synthetic.tracker_sequence(T, seed=8)
    a, b = (PoseTracker.from_yml(*ARMS, n_particles=N, seed=2) for _ in range(2))
    want = _run(a, T, (DeviceArray(imgs), DeviceArray(rois)), True)
    for t in range(T):
        o = b.callback(imgs[t], rois[t])
        assert np.array_equal(o["lml"], want[0][:, t]) and np.array_equal(o["pose"], want[1][t])
        assert np.array_equal(o["tf"].ravel(), want[3][t]) and np.array_equal(o["pose2d"].ravel(), want[4][t])
    a.close()
    b.close()
