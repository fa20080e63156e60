"""Initial tracks written by reset in both state layouts and in a batch, at
the edges of its thread mapping (one particle, a partial block, one past a
block; row counts that do not fill the last group of rows): each track equals
its component's mean and covariance.  The state is held in FP32 in another
basis, so the means and covariances come back to 1e-5 of their norm."""
import numpy as np
import pytest

from mkfbodytracker_pdaf_amd import capi, synthetic
from mkfbodytracker_pdaf_amd.batch import RbpfBatch
from mkfbodytracker_pdaf_amd.rbpf import Rbpf

pytestmark = pytest.mark.gpu


def _check(mdl, bins, x, P):
    mean, cov = mdl.means[bins], mdl.Sigma[bins]
    n = len(bins)
    ex = np.linalg.norm(x - mean, axis=1) / np.linalg.norm(mean, axis=1)
    eP = np.linalg.norm((P - cov).reshape(n, -1), axis=1) / np.linalg.norm(cov.reshape(n, -1), axis=1)
    assert ex.max() < 1e-5 and eP.max() < 1e-5


@pytest.mark.parametrize("N", [1, 63, 256, 257, 1000])
@pytest.mark.parametrize("d", [8, 12, 16, 24])
def test_reset_tracks(N, d):
    mdl = synthetic.make_model(seed=d, d=d)
    bins = np.random.default_rng(N).integers(0, mdl.K, N).astype(np.int32)
    for layout in (capi.PF_LAYOUT_ROWS, capi.PF_LAYOUT_RECORDS):
        if layout == capi.PF_LAYOUT_RECORDS and d > 12:
            continue
        rb = Rbpf(N)
        rb.load_model(mdl.means, mdl.covs, mdl.weights, mdl.gamma, mdl.pca_proj, mdl.pca_mean, sel=mdl.sel, R=mdl.R)
        rb.state_layout = layout
        for b in (bins[::-1].copy(), bins):      # the second reset replaces the first
            rb.reset(b)
        _check(mdl, bins, *rb.get_tracks())
        rb.close()


@pytest.mark.parametrize("d", [12, 24])
def test_reset_batch(d):
    Ns = [1, 257, 700]
    mdl = synthetic.make_model(seed=d, d=d)
    b = RbpfBatch(Ns, [2, 2, 2], K=mdl.K, m=mdl.m, d=d)
    bins = [np.random.default_rng(n).integers(0, mdl.K, n).astype(np.int32) for n in Ns]
    for s in range(3):
        b.load_model(s, mdl.means, mdl.covs, mdl.weights, mdl.gamma, mdl.pca_proj, mdl.pca_mean, mdl.sel, mdl.R)
    for s in range(3):
        b.reset(s, bins[s])
    for s in range(3):
        _check(mdl, bins[s], *b.get_tracks(s))
    b.close()
