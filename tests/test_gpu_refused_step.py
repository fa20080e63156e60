"""A host-driven step that no kernel is compiled for (d = 24 without a selection
basis) is refused after its inputs were sent: the filter's tracks stay, and calls
that follow it at once, with larger exchanges, equal a fresh filter's."""
import numpy as np
import pytest

from mkfbodytracker_pdaf_amd import capi, synthetic
from mkfbodytracker_pdaf_amd.rbpf import Rbpf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [5, 3000])
def test_refused_then_served(N):
    good = synthetic.make_model(seed=4, K=6, d=24)
    bad = synthetic.make_model(seed=4, K=6, d=24)
    bad.pca_proj[:, bad.sel[2:4]] = bad.pca_proj[:, bad.sel[0:2]]
    seq = synthetic.simulate(good, 2, seed=5, cand_per_joint=3, cap=16)
    bins = np.arange(N, dtype=np.int32) % 6
    z = [synthetic.per_particle_measurements(seq.z[t], N, 7 + t) for t in range(2)]

    def load(f, m):
        f.load_model(m.means, m.covs, m.weights, m.gamma, m.pca_proj, m.pca_mean, sel=m.sel, R=m.R)
        f.set_joint_clutter(m.clutter)
        f.reset(bins)

    def serve(f):
        out = [f.step(z[0], 11, 12), f.step_candidates(seq.count[1], seq.cand[1], 13, 14)]
        return [v for _, o in out for v in (o["lw"], o["anc"], o["comp"], o["lml"])] + [f.estimate()]

    f = Rbpf(N)
    load(f, bad)
    before = f.get_tracks()
    for _ in range(3):
        with pytest.raises(capi.PfError):
            f.step_candidates(seq.count[0], seq.cand[0], 1, 2)
        with pytest.raises(capi.PfError):
            f.step(z[1], 3, 4)
    assert all(np.array_equal(p, q) for p, q in zip(f.get_tracks(), before))
    load(f, good)
    g = Rbpf(N)
    load(g, good)
    for p, q in zip(serve(f), serve(g)):
        assert np.array_equal(p, q)
    f.close()
    g.close()
