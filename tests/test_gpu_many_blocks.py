"""Resampling with more than 1024 input blocks of 256 weights, where the
prefix of the block sums is taken once in its own kernel (of the caller's weights,
with 5 x 2^20 pairs of input and output blocks), and, with more than
1700 (1820 at d = 16), the frames of a
device-resident run are step, prefix and ancestor launches: indices bit-exact
against the oracle, and a run equal to host-driven steps bit for bit, on both
sides of both boundaries and at the largest size."""
import numpy as np
import pytest

import oracle
from mkfbodytracker_pdaf_amd import synthetic
from mkfbodytracker_pdaf_amd.devmem import DeviceArray
from mkfbodytracker_pdaf_amd.rbpf import Rbpf

pytestmark = pytest.mark.gpu

EDGE = 262144      # k_prefix above
SPLIT = 435200     # separate launches above
SPLIT16 = 465920   # the same at d = 16


@pytest.mark.parametrize("L", [EDGE, EDGE + 1, 300007, 1 << 20])
@pytest.mark.parametrize("kind", ["even", "few", "one", "zero"])
def test_indices_bit_exact(L, kind):
    rng = np.random.default_rng(L)
    lw = rng.normal(0.0, 2.0, L)
    if kind == "few":          # outputs of one block spread over many input blocks
        lw[rng.random(L) < 0.995] -= 60.0
    elif kind == "one":
        lw[:] = -np.inf
        lw[L - 2] = -1e5
    elif kind == "zero":
        lw[:] = -np.inf
    rb = Rbpf(64)
    for N, u in ((1000, 0), (L, 0xFFFFFFFF), (L - 77, 0x12345678)):
        got, st = rb.resample(lw, N, u, log=True)
        want, wst = oracle.resample_log(lw, N, u)
        assert st == wst == (1 if kind == "zero" else 0)
        assert np.array_equal(got, want)
        w = np.exp(lw - (0.0 if kind == "zero" else lw.max()))
        got, st = rb.resample(w, N, u)
        want, wst = oracle.resample_linear(w, N, u)
        assert st == wst
        assert np.array_equal(got, want)
    rb.close()


@pytest.mark.parametrize("L,blocks", [(1 << 20, 1280), (EDGE + 1, 5115), (600000, 2236)])
def test_callers_weights_both_routes(L, blocks):
    """On both sides of the product of input blocks and blocks of 256 outputs at
    which the prefix gets its own kernel (EDGE + 1 weights are 1025 blocks)."""
    nb = (L + 255) // 256
    assert nb * blocks <= 5 << 20 < nb * (blocks + 1)
    lw = np.random.default_rng(L).normal(0.0, 2.0, L)
    rb = Rbpf(64)
    for N in (256 * blocks, 256 * blocks + 1):
        got, st = rb.resample(lw, N, 0x9E3779B9, log=True)
        want, wst = oracle.resample_log(lw, N, 0x9E3779B9)
        assert st == wst == 0 and np.array_equal(got, want)
    rb.close()


@pytest.mark.parametrize("N,d", [(EDGE, 12), (EDGE + 1, 12), (SPLIT, 12), (SPLIT + 1, 12), (SPLIT + 1, 16),
                                 (SPLIT16, 16), (SPLIT16 + 1, 16)])
def test_run_equals_host_steps(N, d):
    T, cap = 3, 8
    mdl = synthetic.make_model(seed=5, d=d)
    seq = synthetic.simulate(mdl, T, seed=6, cand_per_joint=4, cap=cap)
    bins = oracle.resample_linear(mdl.weights, N, 7)[0]
    d_cnt, d_cand = DeviceArray(seq.count.astype(np.int32)), DeviceArray(seq.cand.astype(np.float32))
    d_uni, d_lml = DeviceArray(seq.uniforms.astype(np.uint32)), DeviceArray.empty(T, np.float64)
    rb = Rbpf(N, cand_capacity=cap)
    rb.load_model(mdl.means, mdl.covs, mdl.weights, mdl.gamma, mdl.pca_proj, mdl.pca_mean, sel=mdl.sel, R=mdl.R)
    rb.set_joint_clutter(mdl.clutter)
    rb.reset(bins)
    want = [rb.step_candidates(seq.count[t], seq.cand[t], int(seq.uniforms[t, 0]), int(seq.uniforms[t, 1]))[1]["lml"]
            for t in range(T)]
    est = rb.estimate()
    for flags in (0, 1):
        rb.reset(bins)
        rb.run_candidates_dev(T, d_cnt.ptr, d_cand.ptr, d_uni.ptr, d_lml.ptr, flags)
        assert rb.synchronize() == 0
        assert rb.last_graph_frames() == (T if flags and N <= (SPLIT16 if d == 16 else SPLIT) else 0)
        assert np.array_equal(d_lml.get(), np.array(want))
        assert np.array_equal(rb.estimate(), est)
    rb.close()
