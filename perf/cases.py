"""What a user of the particle filters has them do, as cases for timing.

Each case is one call path through the public Python interface, over the sizes
that the benchmark, the tests and the evaluation harness use: one filter fed
by a host program frame by frame, recorded sequences replayed from device
memory (shared PDAF detections or one measurement column per particle), the
pose tracker live and on recordings, many ragged sequences at once, the
24-dimensional state, the gradient of the log-marginal-likelihood, and the
plain 2-D filter.
"""
import math
import os

import numpy as np
import torch

from mkfbodytracker_pdaf_amd import capi, synthetic
from mkfbodytracker_pdaf_amd.batch import RbpfBatch
from mkfbodytracker_pdaf_amd.pf2d import Pf2d
from mkfbodytracker_pdaf_amd.rbpf import Rbpf
from mkfbodytracker_pdaf_amd.torch_adjoint import BatchProblem, lml as lml_of
from mkfbodytracker_pdaf_amd.tracker import PoseTracker

CAP = 16                                  # detections per joint the filters are created for
P_DETECT, GATE = 0.95, 9.210340371976184  # the library's defaults
FIVE = ("head", "left_hand", "right_hand", "left_elbow", "right_elbow")
ARMS = tuple(os.path.join("tests", "golden", "data%s_PCA_100000_15_12.yml" % a) for a in ("13D", "23D"))
POSE = 22                                 # length of the shipped models' pose vector


def listed():
    return [
        # the reference's operating point: 500 particles, one 6 x N measurement from the host per camera frame
        {"name": "live_500", "kind": "live", "n": 500, "d": 12, "mode": "ref"},
        # the whole tracker called once per camera image, 500 particles and 5,000 proposals per arm
        {"name": "live_tracker_500", "kind": "live_tracker", "n": 500},
        # a short recording through a small filter, 4 detections per hand
        {"name": "replay_1k", "kind": "replay", "n": 1000, "t": 300, "d": 12, "det": 4},
        # the benchmark's headline: 100,000 particles, 8 detections per hand
        {"name": "replay_100k", "kind": "replay", "n": 100000, "t": 200, "d": 12, "det": 8},
        # as many particles as one filter takes, to the nearest odd thousand
        {"name": "replay_1m", "kind": "replay", "n": 1000003, "t": 24, "d": 12, "det": 8},
        # recorded per-particle measurements (the reference's form of the update)
        {"name": "replay_measured_20k", "kind": "measured", "n": 20011, "t": 100, "d": 12},
        # a recording through the tracker at the reference's size, and at the benchmark's
        {"name": "tracker_500", "kind": "tracker", "n": 500, "t": 48},
        {"name": "tracker_100k", "kind": "tracker", "n": 100000, "t": 32},
        # ragged recordings advanced together, each with its own model
        {"name": "batch_ragged", "kind": "batch", "s": 64, "n_lo": 1000, "n_hi": 64000, "t_lo": 10, "t_hi": 100,
         "d": 12, "k": 15, "det": 8},
        # the scaled state: 24 dimensions, 64 components, 5 PDAF joints
        {"name": "batch_d24", "kind": "batch", "s": 32, "n_lo": 31250, "n_hi": 31250, "t_lo": 8, "t_hi": 8,
         "d": 24, "k": 64, "det": 11},
        # one training step on the model's parameters
        {"name": "gradient", "kind": "gradient", "s": 16, "n": 16384, "t": 60, "every": 50},
        # the plain 2-D filter, one update with host measurements and noise
        {"name": "plain_20k", "kind": "plain", "n": 20000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("live", "live_tracker", "replay", "replay", "replay", "measured", "tracker", "tracker", "batch",
                       "batch", "gradient", "plain"))
    if kind == "live":
        return {"kind": kind, "n": _log(rng, 200, 20000), "d": rng.choice((8, 12, 12, 16)),
                "mode": rng.choice(("ref", "cand"))}
    if kind == "live_tracker":
        return {"kind": kind, "n": _log(rng, 200, 20000)}
    if kind == "replay":
        n = _log(rng, 500, 1048576)
        return {"kind": kind, "n": n, "t": max(8, min(rng.randint(100, 400), 24000000 // n)),
                "d": rng.choice((8, 12, 12, 16)), "det": rng.choice((4, 8))}
    if kind == "measured":
        n = _log(rng, 500, 200000)
        return {"kind": kind, "n": n, "t": max(8, min(rng.randint(30, 100), 3000000 // n)), "d": rng.choice((8, 12, 16))}
    if kind == "tracker":
        return {"kind": kind, "n": _log(rng, 300, 100000), "t": rng.randint(17, 48)}
    if kind == "batch" and rng.random() < 0.4:
        s, n = rng.randint(4, 32), _log(rng, 2000, 31250)
        return {"kind": kind, "s": s, "n_lo": n, "n_hi": n, "t_lo": 4, "t_hi": rng.randint(5, 8), "d": 24,
                "k": rng.choice((15, 64)), "det": 11}
    if kind == "batch":
        return {"kind": kind, "s": rng.randint(2, 64), "n_lo": 1000, "n_hi": _log(rng, 4000, 64000), "t_lo": 10,
                "t_hi": rng.randint(20, 100), "d": 12, "k": 15, "det": rng.choice((4, 8))}
    if kind == "gradient":
        return {"kind": kind, "s": rng.randint(1, 16), "n": _log(rng, 500, 16384), "t": rng.randint(10, 60),
                "every": rng.choice((10, 25, 50))}
    return {"kind": kind, "n": _log(rng, 500, 50000)}


# ---------------------------------------------------------------- inputs
def _model(case, seed):
    if case.get("d") == 24:
        return synthetic.make_model(seed=seed, K=case["k"], d=24, joints=FIVE, clutter=(1, 1, 1, 1, 1))
    return synthetic.make_model(seed=seed, K=case.get("k", 15), d=case.get("d", 12))


def _lam(det):
    """Clutter density of det detections per joint and image, one of them true."""
    return (det - 1) / (640.0 * 480.0)


def _first_uniform(seed):
    return int(capi.philox_u32(seed, 2, 0, 1)[0])


def _gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _filter(n, mdl, det):
    f = Rbpf(n, cand_capacity=CAP, clutter_density=_lam(det))
    f.load_model(mdl.means, mdl.covs, mdl.weights, mdl.gamma, mdl.pca_proj, mdl.pca_mean, sel=mdl.sel, R=mdl.R)
    f.set_joint_clutter(mdl.clutter)
    return f


def _bins(f, mdl, n, seed):
    return f.resample(mdl.weights, n, _first_uniform(seed))[0]


def _measurements(mdl, n, t, seed):
    """t frames of m x n measurement columns and their uniforms (host)."""
    seq = synthetic.simulate_fast(mdl, t, seed)
    z = np.stack([synthetic.per_particle_measurements(seq.z[i], n, seed + 7 * i) for i in range(t)])
    return z, seq.uniforms


def _detections(mdl, t, det, seed):
    seq = synthetic.simulate_fast(mdl, t, seed, cand_per_joint=det, cap=CAP)
    return seq.count.astype(np.int32), seq.cand.astype(np.float32), seq.uniforms.astype(np.uint32).view(np.int32)


LIVE_FRAMES = 16


def _live_inputs(case, seed):
    mdl = _model(case, seed)
    if case["mode"] == "ref":
        return mdl, _measurements(mdl, case["n"], LIVE_FRAMES, seed)
    seq = synthetic.simulate_fast(mdl, LIVE_FRAMES, seed, cand_per_joint=8, cap=CAP)
    return mdl, (seq.count, seq.cand, seq.uniforms)


def _batch_sizes(case):
    """Particle counts (log-uniform) and lengths (uniform) of a batch's sequences."""
    rng = np.random.default_rng([case["s"], case["n_hi"], case["t_hi"]])
    ns = np.exp(rng.uniform(math.log(case["n_lo"]), math.log(case["n_hi"]), case["s"]) + 1e-9).astype(np.int32)
    return ns, rng.integers(case["t_lo"], case["t_hi"] + 1, case["s"]).astype(np.int32)


def _plain_inputs(case, seed):
    """A GMM over the 8 pixel coordinates, particles around it, and 4 frames
    of measurements (row 0: the tracked hand, row 1: the head)."""
    rng = np.random.default_rng(seed)
    n, k = case["n"], 10
    home = np.array([320.0, 80.0, 320.0, 150.0, 240.0, 200.0, 200.0, 280.0])
    means = home + 30.0 * rng.standard_normal((k, 8))
    a = 12.0 * rng.standard_normal((k, 8, 8))
    covs = a @ a.transpose(0, 2, 1) + 400.0 * np.eye(8)
    start = home + 15.0 * rng.standard_normal((n, 8))
    frames = [{"meas": np.stack([home[6:8], home[0:2]]) + 8.0 * rng.standard_normal((2, 2)),
               "u": int(rng.integers(0, 2 ** 32)), "normals": rng.standard_normal((n, 8)),
               "reinit": rng.random((n, 8))} for _ in range(4)]
    return means, covs, rng.dirichlet(np.full(k, 5.0)), start, frames


def prepare(case, seed):
    kind = case["kind"]
    st = {"kind": kind, "case": case, "at": 0}
    if kind == "live":
        mdl, st["inputs"] = _live_inputs(case, seed)
        f = _filter(case["n"], mdl, 8)
        f.reset(_bins(f, mdl, case["n"], seed))
        st["filter"] = f
    elif kind in ("live_tracker", "tracker"):
        t = case.get("t", LIVE_FRAMES)
        imgs, rois = synthetic.tracker_sequence(t, seed=seed)
        st["tracker"] = PoseTracker.from_yml(ARMS[0], ARMS[1], n_particles=case["n"], seed=seed)
        if kind == "live_tracker":
            st["imgs"], st["rois"] = imgs, rois
        else:
            st["imgs"], st["rois"] = _gpu(imgs), _gpu(rois)
            st["bins"] = [arm.resample(capi.yml_read_matrix(path, "weights").ravel(), case["n"],
                                       _first_uniform(seed + a))[0]
                          for a, (arm, path) in enumerate(zip(st["tracker"].arms, ARMS))]
            f64 = dict(dtype=torch.float64, device="cuda")
            st["out"] = {"lml": torch.zeros(2, t, **f64), "pose": torch.zeros(t, 2, POSE, **f64),
                         "pos3d": torch.zeros(t, 2, 3, 5, **f64), "tf": torch.zeros(t, 8, 3, **f64),
                         "pose2d": torch.zeros(t, 8, 2, **f64)}
    elif kind in ("replay", "measured"):
        mdl = _model(case, seed)
        n, t = case["n"], case["t"]
        f = _filter(n, mdl, case.get("det", 8))
        st["filter"], st["bins"] = f, _bins(f, mdl, n, seed)
        if kind == "replay":
            st["count"], st["cand"], uni = (_gpu(a) for a in _detections(mdl, t, case["det"], seed))
        else:
            seq = synthetic.simulate_fast(mdl, t, seed)
            gen = torch.Generator(device="cuda").manual_seed(seed)
            z = torch.randn(t, mdl.m, n, generator=gen, device="cuda")
            st["z"] = z.mul_(5.0).add_(_gpu(seq.z.astype(np.float32))[:, :, None])
            uni = _gpu(seq.uniforms.astype(np.uint32).view(np.int32))
        st["uni"], st["lml"] = uni, torch.zeros(t, dtype=torch.float64, device="cuda")
    elif kind == "batch":
        ns, ts = _batch_sizes(case)
        models = [_model(case, seed + 1000 * i) for i in range(case["s"])]
        b = RbpfBatch(ns, ts, K=case["k"], m=models[0].m, d=case["d"], cand_capacity=CAP,
                      clutter_density=_lam(case["det"]))
        for i, m in enumerate(models):
            b.load_model(i, m.means, m.covs, m.weights, m.gamma, m.pca_proj, m.pca_mean, m.sel, m.R)
        b.set_joint_clutter(models[0].clutter)
        helper = Rbpf(1)
        st["bins"] = [_bins(helper, models[i], int(ns[i]), seed + i) for i in range(case["s"])]
        helper.close()
        seqs = [_detections(models[i], int(ts[i]), case["det"], seed + i) for i in range(case["s"])]
        st["batch"] = b
        st["count"], st["cand"], st["uni"] = (_gpu(np.concatenate(a)) for a in zip(*seqs))
        st["lml"] = torch.zeros(int(ts.sum()), dtype=torch.float64, device="cuda")
    elif kind == "gradient":
        mdl = _model(case, seed)
        s, n, t = case["s"], case["n"], case["t"]
        seqs = [_detections(mdl, t, 8, seed + i) for i in range(s)]
        helper = Rbpf(1)
        bins = [_bins(helper, mdl, n, seed + i) for i in range(s)]
        helper.close()
        st["problem"] = BatchProblem([n] * s, [t] * s, mdl.pca_proj, mdl.pca_mean, mdl.sel, mdl.R, mdl.clutter,
                                     *(np.concatenate(a) for a in zip(*seqs)), bins,
                                     checkpoint_every=case["every"], cand_capacity=CAP, clutter_density=_lam(8))
        st["params"] = [torch.from_numpy(np.ascontiguousarray(a)).requires_grad_() for a in (
            mdl.means, np.log(mdl.weights), 1.0 - mdl.gamma, np.linalg.cholesky(mdl.Sigma))]
    else:
        means, covs, weights, start, st["frames"] = _plain_inputs(case, seed)
        f = Pf2d(case["n"])
        f.load_gmm(means, covs, weights)
        f.set_particles(start)
        st["filter"] = f
    torch.cuda.synchronize()
    return st


# ------------------------------------------------------------------ passes
def run(st):
    kind, case = st["kind"], st["case"]
    if kind == "live":                    # the next camera frame through one filter, and the pose estimate
        i = st["at"] % LIVE_FRAMES
        st["at"] += 1
        f = st["filter"]
        if case["mode"] == "ref":
            z, uni = st["inputs"]
            _, out = f.step(z[i], int(uni[i, 0]), int(uni[i, 1]))
        else:
            count, cand, uni = st["inputs"]
            _, out = f.step_candidates(count[i], cand[i], int(uni[i, 0]), int(uni[i, 1]))
        return [out["lw"], out["lml"], out["comp"], out["anc"], f.estimate()]
    if kind == "live_tracker":            # the next camera image through the tracker
        i = st["at"] % LIVE_FRAMES
        st["at"] += 1
        out = st["tracker"].callback(st["imgs"][i], st["rois"][i])
        return [out["lml"], out["pose"], out["pos3d"], out["tf"], out["pose2d"]]
    if kind == "tracker":                 # a recording from its first image
        tr, o = st["tracker"], st["out"]
        for arm, bins in zip(tr.arms, st["bins"]):
            arm.reset(bins)
        tr.reset()
        tr.run_dev(case["t"], st["imgs"].data_ptr(), st["rois"].data_ptr(), o["lml"].data_ptr(), o["pose"].data_ptr(),
                   o["pos3d"].data_ptr(), o["tf"].data_ptr(), o["pose2d"].data_ptr())
        tr.synchronize()
        return o
    if kind in ("replay", "measured"):    # a recording from the initial tracks to its last pose estimate
        f = st["filter"]
        f.reset(st["bins"])
        if kind == "replay":
            f.run_candidates_dev(case["t"], st["count"].data_ptr(), st["cand"].data_ptr(), st["uni"].data_ptr(),
                                 st["lml"].data_ptr())
        else:
            f.run_ref_dev(case["t"], st["z"].data_ptr(), st["uni"].data_ptr(), st["lml"].data_ptr())
        return [st["lml"], f.estimate()]
    if kind == "batch":                   # every recording from its initial tracks to its last pose estimate
        b = st["batch"]
        for i, bins in enumerate(st["bins"]):
            b.reset(i, bins)
        b.run_dev(st["count"].data_ptr(), st["cand"].data_ptr(), st["uni"].data_ptr(), st["lml"].data_ptr())
        return [st["lml"], np.stack([b.estimate(i) for i in range(b.S)])]
    if kind == "gradient":                # the loss and its gradients by backward()
        for p in st["params"]:
            p.grad = None
        value = lml_of(*st["params"], st["problem"])
        value.backward()
        return [value.detach()] + [p.grad for p in st["params"]]
    f, frame = st["filter"], st["frames"][st["at"] % len(st["frames"])]
    st["at"] += 1
    _, out = f.update(frame["meas"], frame["u"], frame["normals"], frame["reinit"])
    return [out["lw"], out["anc"], f.estimate()]


# ------------------------------------------------------------------- work
def _step_work(n, d, m, det, measured):
    """One filter frame of n particles: the ancestor's x and packed P read,
    the new ones written, the log-weight written and the ancestor read; the
    predict, m/2 two-row updates (each the innovation, its gain and the
    rank-2 update of packed P) and det detections per joint of about 20
    operations each."""
    p = d * (d + 1) // 2
    b = 8 * (d + p) + 8 + (4 * m if measured else 0)
    f = 2 * (d + p) + (m // 2) * (4 * p + 10 * d + 40) + (m // 2) * det * 20
    return n * b, n * f


def work(case):
    kind, n, d = case["kind"], case.get("n", 0), case.get("d", 12)
    if kind == "live":
        b, f = _step_work(n, d, 6, 1 if case["mode"] == "ref" else 8, case["mode"] == "ref")
        return {"bytes": b + 12 * n, "flops": f}
    if kind in ("live_tracker", "tracker"):
        # per arm: 10 n proposals weighted (about 300 operations each) and their weights
        # written and read, the filter frame, the estimate of the resampled states; one image
        b, f = _step_work(n, 12, 6, 1, True)
        t = case.get("t", 1)
        return {"bytes": t * (2 * (b + 160 * n + 48 * n) + 480 * 640), "flops": t * (2 * (f + 3000 * n) + 480 * 640 * 60)}
    if kind in ("replay", "measured"):
        b, f = _step_work(n, d, 6, case.get("det", 1), kind == "measured")
        return {"bytes": case["t"] * b, "flops": case["t"] * f}
    if kind == "batch":
        ns, ts = _batch_sizes(case)
        b, f = _step_work(1, d, 10 if d == 24 else 6, case["det"], False)
        pf = float((ns.astype(np.float64) * ts).sum())
        return {"bytes": b * pf, "flops": f * pf}
    if kind == "gradient":
        # forward, then per frame the state read again with its adjoint read and written
        b, f = _step_work(n, 12, 6, 8, False)
        k = case["s"] * case["t"]
        return {"bytes": k * (2 * b + n * 12 * (12 + 78) + 8 * n), "flops": 4 * k * f}
    # 10 components of an 8-dimensional density, the state and the noise read, the state written
    return {"bytes": n * (32 + 64 + 32 + 8), "flops": n * 10 * 160}


# ------------------------------------------------------ plain 64-bit values
def _systematic(w, n, u):
    """Systematic resampling of weights w into n indices, uniform u / 2^32."""
    c = np.cumsum(w)
    pos = (np.arange(n) + u / 2.0 ** 32) * (c[-1] / n)
    return np.minimum(np.searchsorted(c, pos, side="right"), len(w) - 1)


def _joint(x, P, h, bh, r):
    """Innovation of one two-row joint: (y, S, H P)."""
    hp = np.einsum("ij,njk->nik", h, P)
    return x @ h.T + bh, hp @ h.T + r, hp


def _frame64(mdl, x, P, u, z=None, count=None, cand=None, lam=None):
    """One frame in 64 bits: (log-weights, components, x, P) before resampling."""
    n, d = x.shape
    k = _systematic(mdl.weights, n, u)
    g = mdl.gamma[k]
    x = g[:, None] * x + (1 - g)[:, None] * mdl.means[k]
    P = (g * g)[:, None, None] * P + (1 - g * g)[:, None, None] * mdl.Sigma[k]
    H, BH = mdl.H(), mdl.BH()
    lw = np.zeros(n)
    joints = range(mdl.m // 2)
    if z is None:
        joints = sorted(joints, key=lambda b: bool(mdl.clutter[b]))
    for b in joints:
        rows = slice(2 * b, 2 * b + 2)
        y, S, hp = _joint(x, P, H[rows], BH[rows], mdl.R[rows, rows])
        Si = np.linalg.inv(S)
        logn = -0.5 * np.log(np.linalg.det(S)) - math.log(2 * math.pi)
        K = np.einsum("nik,nij->nkj", hp, Si)
        if z is not None or not mdl.clutter[b]:
            if z is None and count[b] == 0:
                continue
            nu = (z[rows].T if z is not None else cand[b, 0]) - y
            lw += logn - 0.5 * np.einsum("ni,nij,nj->n", nu, Si, nu)
            x = x + np.einsum("nki,ni->nk", K, nu)
            P = P - K @ hp
            continue
        nu = cand[b, None, : count[b]] - y[:, None]
        d2 = np.einsum("nci,nij,ncj->nc", nu, Si, nu)
        e = np.where(d2 <= GATE, P_DETECT / lam * np.exp(logn[:, None] - 0.5 * d2), 0.0)
        ell = 1.0 - P_DETECT * (1.0 - math.exp(-0.5 * GATE)) + e.sum(1)
        beta = e / ell[:, None]
        v = np.einsum("nc,nci->ni", beta, nu)
        spread = np.einsum("nc,nci,ncj->nij", beta, nu, nu) - v[:, :, None] * v[:, None, :]
        lw += np.log(ell)
        x = x + np.einsum("nki,ni->nk", K, v)
        P = P - beta.sum(1)[:, None, None] * (K @ hp) + K @ spread @ K.transpose(0, 2, 1)
    return lw, k, x, 0.5 * (P + P.transpose(0, 2, 1))


def _log_mean(lw):
    m = lw.max()
    return m + math.log(np.exp(lw - m).mean())


def exact(case, seed):
    kind = case["kind"]
    if kind == "live":
        mdl, inputs = _live_inputs(case, seed)
        b = _systematic(mdl.weights, case["n"], _first_uniform(seed))
        uni = inputs[-1]
        how = {"z": inputs[0][0]} if case["mode"] == "ref" else {"count": inputs[0][0], "cand": inputs[1][0],
                                                                 "lam": _lam(8)}
        lw, _, x, _ = _frame64(mdl, mdl.means[b], mdl.Sigma[b], int(uni[0, 0]), **how)
        a = _systematic(np.exp(lw - lw.max()), case["n"], int(uni[0, 1]))
        return [lw, _log_mean(lw), None, None, x[a].mean(0)]
    if kind == "replay" and case["n"] * case["t"] <= 400000:
        mdl = _model(case, seed)
        count, cand, uni = _detections(mdl, case["t"], case["det"], seed)
        b = _systematic(mdl.weights, case["n"], _first_uniform(seed))
        x, P, out = mdl.means[b], mdl.Sigma[b], []
        for i in range(case["t"]):
            lw, _, x, P = _frame64(mdl, x, P, int(uni[i, 0]) & 0xffffffff, count=count[i], cand=cand[i].astype(np.float64),
                                   lam=_lam(case["det"]))
            a = _systematic(np.exp(lw - lw.max()), case["n"], int(uni[i, 1]) & 0xffffffff)
            x, P = x[a], P[a]
            out.append(_log_mean(lw))
        return [np.array(out), x.mean(0)]
    if kind == "plain":
        means, covs, weights, start, frames = _plain_inputs(case, seed)
        z = frames[0]["meas"]
        dev = start[:, None] - means
        q = np.einsum("nki,kij,nkj->nk", dev, np.linalg.inv(covs), dev)
        comp = np.log(weights) - 0.5 * (8 * math.log(2 * math.pi) + np.linalg.slogdet(covs)[1]) - 0.5 * q
        top = comp.max(1, keepdims=True)
        lw = top[:, 0] + np.log(np.exp(comp - top).sum(1))
        for row, at in ((z[0], start[:, 6:8]), (z[1], start[:, 0:2])):
            lw = lw - 0.5 * ((row - at) ** 2).sum(1) / 15.0 - math.log(2 * math.pi * 15.0)
        return [lw, None, None]
    return None  # long runs: each frame's draws depend on every rounding of the frames before it
