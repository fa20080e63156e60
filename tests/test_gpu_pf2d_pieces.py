"""Plain-filter updates whose random walk goes to the device in pieces of at
least 4096 particles (up to four) while the frame is resampled, or, above
16 MiB of steps and outputs, by copies: the moved particles exact in FP32, the
ancestors bit-exact, a degenerate update re-drawn and the next one ordinary."""
import numpy as np
import pytest

import oracle
from mkfbodytracker_pdaf_amd.capi import check, f64, ptr
from mkfbodytracker_pdaf_amd.pf2d import Pf2d

pytestmark = pytest.mark.gpu

LIMIT = (16 << 20) // 40        # 8 steps and two outputs of 4 bytes per particle
COLS = [2, 3, 4, 5, 6, 7, 0, 1]


@pytest.mark.parametrize("N", [1, 4096, 4097, 8191, 16385, 20000, LIMIT, LIMIT + 1])
def test_walk(gpu, N):
    rng = np.random.default_rng(N)
    mu = rng.uniform(100, 400, (4, 8))
    g = Pf2d(N, 8, side=1)
    g.load_gmm(mu, np.stack([np.diag(rng.uniform(400, 4000, 8)) for _ in range(4)]), rng.dirichlet(np.ones(4)))
    reinit = rng.random((N, 8))
    g.init(reinit)
    meas = np.array([[400.0, 200.0], [100.0, 300.0]])
    for t in range(4):
        if t == 2:                                   # no usable weight: re-drawn
            g.set_particles(np.full((N, 8), np.nan))
        pin = g.get_particles()[0].astype(np.float32)
        normals, U = rng.standard_normal((N, 8)), int(rng.integers(0, 2 ** 32))
        if t == 3:                                   # outputs left out
            st = check(g.lib.pf2d_update(g.h, ptr(f64(meas)), U, ptr(normals), ptr(reinit), None, None))
            out = None
        else:
            st, out = g.update(meas, U, normals, reinit)
        assert st == (1 if t == 2 else 0)
        got, wts = g.get_particles()
        if t == 2:
            base = oracle.pf2d_init(N, 8, 1, reinit).astype(np.float32)
            assert np.allclose(wts, 1.0 / N)
        elif t < 3:
            want, _ = oracle.resample_log(out["lw"].astype(np.float64), N, U)
            assert np.array_equal(out["anc"], want)
            base = pin[want].copy()
        else:
            continue
        base[:, COLS] += (5.0 * normals).astype(np.float32)
        if t == 2:                                   # the FP32 bounds' rounding differs by an ulp
            assert np.allclose(got, base, rtol=1e-6, atol=1e-4)
        else:
            assert np.array_equal(got, base.astype(np.float64))
        e = g.estimate()
        assert np.allclose(e, oracle.pf2d_estimate(got, wts), rtol=1e-9, atol=1e-6)
    g.close()
