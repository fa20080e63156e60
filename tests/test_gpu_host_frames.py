"""Host-driven frames, whose data goes through one pinned buffer up to 4 MiB
and by copies above: every output equal bit for bit to the device's own values
(a device-resident run, and the same frames with other block sizes and with
outputs left out) and the ancestors bit-exact against the oracle, at one
particle, around a block, and on both sides of the buffer's limit."""
import numpy as np
import pytest

import oracle
from mkfbodytracker_pdaf_amd import synthetic
from mkfbodytracker_pdaf_amd.capi import check, i32, f64, ptr
from mkfbodytracker_pdaf_amd.devmem import DeviceArray
from mkfbodytracker_pdaf_amd.rbpf import Rbpf

pytestmark = pytest.mark.gpu

T = 3
# 24 bytes of measurement and 12 of outputs per particle
LIMIT = ((4 << 20) - 16) // 36


def open_filter(mdl, N, bins, **cfg):
    rb = Rbpf(N, **cfg)
    rb.load_model(mdl.means, mdl.covs, mdl.weights, mdl.gamma, mdl.pca_proj, mdl.pca_mean, sel=mdl.sel, R=mdl.R)
    rb.reset(bins)
    return rb


@pytest.mark.parametrize("N", [1, 255, 257, 1001, LIMIT, LIMIT + 1])
@pytest.mark.parametrize("mode", ["ref", "cand"])
def test_host_frames(N, mode):
    mdl = synthetic.make_model(seed=5)
    m = len(mdl.sel)
    seq = synthetic.simulate(mdl, T, seed=6, cand_per_joint=4, cap=16)
    rng = np.random.default_rng(N)
    Z = rng.normal(300.0, 40.0, (T, m, N)).astype(np.float32)
    bins = oracle.resample_linear(mdl.weights, N, 7)[0]
    uni = seq.uniforms.astype(np.uint32)

    def frame(rb, t, outputs=True):
        u = int(uni[t, 0]), int(uni[t, 1])
        if outputs:
            return rb.step(Z[t], *u) if mode == "ref" else rb.step_candidates(seq.count[t], seq.cand[t], *u)
        if mode == "ref":
            return check(rb.lib.pf_step(rb.h, ptr(f64(Z[t])), *u, None, None, None, None)), None
        return check(rb.lib.pf_step_candidates(rb.h, ptr(i32(seq.count[t])), ptr(f64(seq.cand[t])), *u, None, None,
                                               None, None)), None

    rb = open_filter(mdl, N, bins)
    outs, ests = [], []
    for t in range(T):
        st, out = frame(rb, t)
        want, wst = oracle.resample_log(out["lw"].astype(np.float64), N, int(uni[t, 1]))
        assert st == wst == 0
        assert np.array_equal(out["anc"], want)
        assert out["comp"].min() >= 0 and out["comp"].max() < rb.K
        outs.append(out)
        ests.append(rb.estimate())
    # a frame whose weights are all zero reports it, once
    if mode == "ref":
        st, out = rb.step(np.full((m, N), 1e30), 1, 2)
        assert st == 1 and np.array_equal(out["anc"], np.arange(N))
    rb.reset(bins)
    for t in range(T):
        st, _ = frame(rb, t, outputs=False)
        assert st == 0
        assert np.array_equal(rb.estimate(), ests[t])
    d_uni, d_lml = DeviceArray(uni), DeviceArray.empty(T, np.float64)
    rb.reset(bins)
    if mode == "ref":
        d_z = DeviceArray(Z)
        rb.run_ref_dev(T, d_z.ptr, d_uni.ptr, d_lml.ptr)
    else:
        d_cnt, d_cand = DeviceArray(seq.count.astype(np.int32)), DeviceArray(seq.cand.astype(np.float32))
        rb.run_candidates_dev(T, d_cnt.ptr, d_cand.ptr, d_uni.ptr, d_lml.ptr)
    assert rb.synchronize() == 0
    assert np.array_equal(d_lml.get(), np.array([o["lml"] for o in outs]))
    assert np.array_equal(rb.estimate(), ests[-1])
    rb.close()
    # blocks other than the resampler's: the weights are taken in their own launch
    rb = open_filter(mdl, N, bins, block_size=128)
    for t in range(T):
        st, out = frame(rb, t)
        assert st == 0
        for k in ("lw", "anc", "comp", "lml"):
            assert np.array_equal(out[k], outs[t][k])
    rb.close()
