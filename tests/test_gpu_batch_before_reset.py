"""Reads of a batch whose models are loaded but whose tracks were never set: the
values are unspecified, but every particle's ancestor index is valid."""
import numpy as np
import pytest

from mkfbodytracker_pdaf_amd import synthetic
from mkfbodytracker_pdaf_amd.batch import RbpfBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [12, 24])
def test_reads_before_the_first_reset(d):
    N = 700
    m = synthetic.make_model(seed=2, K=4, d=d, clutter=(1, 1, 1))
    b = RbpfBatch([N], [3], K=4, m=6, d=d, cand_capacity=8)
    b.load_model(0, m.means, m.covs, m.weights, m.gamma, m.pca_proj, m.pca_mean, m.sel, m.R)
    assert not b.last_frame(0)[1].any()
    x, P = b.get_tracks(0)
    assert x.shape == (N, d) and P.shape == (N, d, d) and b.estimate(0).shape == (d,)
    b.close()
