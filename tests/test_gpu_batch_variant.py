"""Changing the d = 24 batch's kernel: before any tracks it only selects the
kernel (no conversion, the schedule's tile size included), afterwards the tracks
move to the other layout bit for bit, from either state buffer (a recording of
odd length ends in the second), and a change and back changes nothing.  Imported
tracks are the same bits in both layouts."""
import numpy as np
import pytest

import oracle
from mkfbodytracker_pdaf_amd import capi, synthetic
from mkfbodytracker_pdaf_amd.batch import RbpfBatch
from mkfbodytracker_pdaf_amd.devmem import DeviceArray

pytestmark = pytest.mark.gpu

ROWS, QUAD, MFMA = capi.PF_BATCH_VALU, capi.PF_BATCH_QUAD_VALU, capi.PF_BATCH_MFMA
NS, TS, K = [70, 513, 1], [3, 2, 1], 9


def _batch():
    models = [synthetic.make_model(seed=7 + s, K=K, d=24, clutter=(1, 1, 1)) for s in range(len(NS))]
    seqs = [synthetic.simulate(models[s], TS[s], seed=30 + s, cand_per_joint=5, cap=8) for s in range(len(NS))]
    bins = [oracle.resample_linear(models[s].weights, NS[s], 40 + s)[0] for s in range(len(NS))]
    b = RbpfBatch(NS, TS, K=K, m=6, d=24, cand_capacity=8)
    dev = [DeviceArray(np.concatenate([getattr(q, f) for q in seqs]).astype(t))
           for f, t in (("count", np.int32), ("cand", np.float32), ("uniforms", np.uint32))]
    return b, models, bins, dev


def _load(b, models):
    for s, m in enumerate(models):
        b.load_model(s, m.means, m.covs, m.weights, m.gamma, m.pca_proj, m.pca_mean, m.sel, m.R)
    b.set_joint_clutter(models[0].clutter)


def _state(b):
    return [v for s in range(len(NS)) for v in b.get_tracks(s) + (b.estimate(s),)]


@pytest.mark.parametrize("variant", [QUAD, MFMA])
def test_change_of_kernel(variant):
    b, models, bins, dev = _batch()
    lml = DeviceArray.empty(sum(TS), np.float64)
    # without tracks, from a schedule of another tile size
    b.variant = ROWS
    b.schedule = (64, 1, 3)
    b.variant = variant
    assert b.variant == variant and tuple(b.schedule) == (256, 1, 3)
    _load(b, models)
    b.variant = ROWS
    b.variant = variant
    for s, bi in enumerate(bins):
        b.reset(s, bi)
    b.run_dev(*(d.ptr for d in dev), lml.ptr)
    want, want_lml = _state(b), lml.get()
    for v in (ROWS, variant, ROWS):
        b.variant = v
        assert all(np.array_equal(p, q) for p, q in zip(_state(b), want))
    # reset as rows, run as records
    for s, bi in enumerate(bins):
        b.reset(s, bi)
    b.variant = variant
    b.run_dev(*(d.ptr for d in dev), lml.ptr)
    assert np.array_equal(lml.get(), want_lml)
    assert all(np.array_equal(p, q) for p, q in zip(_state(b), want))
    b.close()


@pytest.mark.parametrize("variant", [QUAD, MFMA])
def test_imported_tracks(variant):
    """The import's FP64 products and FP32 rounding do not depend on the
    layout, nor does the export of what it stored (sequences of even length:
    the initial tracks' buffer is the one read)."""
    b, models, bins, _ = _batch()
    _load(b, models)
    even = [s for s in range(len(NS)) if TS[s] % 2 == 0]
    got = []
    for v in (ROWS, variant):
        b.variant = v
        for s in range(len(NS)):
            a = np.random.default_rng(s).standard_normal((NS[s], 24, 24))
            b.set_tracks(s, np.random.default_rng(9 + s).standard_normal((NS[s], 24)),
                         a @ a.transpose(0, 2, 1) + np.eye(24))
        got.append([q for s in even for q in b.get_tracks(s) + (b.estimate(s),)])
    assert even and all(np.array_equal(p, q) for p, q in zip(*got))
    b.close()
