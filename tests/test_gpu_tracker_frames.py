"""Host-driven tracker frames, whose image and ROI are read from and whose
outputs are written to pinned memory: equal to a device-resident run of the
same frames for images that do not fill whole 16-byte words, and the arms'
first estimates (one launch pair for both) equal to each arm's own."""
import os

import numpy as np
import pytest

from mkfbodytracker_pdaf_amd import synthetic
from mkfbodytracker_pdaf_amd.devmem import DeviceArray
from mkfbodytracker_pdaf_amd.tracker import PoseTracker

pytestmark = pytest.mark.gpu

ARMS = [os.path.join(os.path.dirname(__file__), "golden", f"data{a}_PCA_100000_15_12.yml") for a in ("13D", "23D")]


@pytest.mark.parametrize("rows,cols", [(480, 640), (47, 61), (33, 32), (17, 99)])
@pytest.mark.parametrize("N", [1, 257])
def test_frames_equal_run(rows, cols, N):
    T = 4
    imgs, rois = synthetic.tracker_sequence(T, seed=8, rows=rows, cols=cols)
    a, b = (PoseTracker.from_yml(*ARMS, n_particles=N, seed=2, rows=rows, cols=cols) for _ in range(2))
    dev = DeviceArray(imgs), DeviceArray(rois)
    out = [DeviceArray.empty(s, np.float64) for s in ((2, T), (T, 2, 22), (T, 2, 15), (T, 24), (T, 16))]
    a.run_dev(T, dev[0].ptr, dev[1].ptr, *(o.ptr for o in out))
    a.synchronize()
    want = [o.get() for o in out]
    for t in range(T):
        o = b.callback(imgs[t], rois[t])
        assert np.array_equal(o["lml"], want[0][:, t]) and np.array_equal(o["pose"], want[1][t])
        assert np.array_equal(o["pos3d"].ravel(), want[2][t].ravel())
        assert np.array_equal(o["tf"].ravel(), want[3][t]) and np.array_equal(o["pose2d"].ravel(), want[4][t])
    la, lb = a.get_last(), b.get_last()
    for k in ("blurred", "bins", "Z"):
        assert np.array_equal(la[k], lb[k])
    p = b.pose()
    assert np.array_equal(p["pose"], o["pose"])
    # both arms' estimates are each arm's own (FP64 sums of 12 products: 1e-12)
    for i, arm in enumerate(b.arms):
        own = arm.estimate() @ b.pca_proj[i] + b.pca_mean[i]
        assert np.allclose(own, p["pose"][i], rtol=1e-12, atol=1e-10)
    a.close()
    b.close()
