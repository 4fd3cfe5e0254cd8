"""Performance cases of the discretization library.

Each case is one call (or one short sequence of calls) that a user of the
library makes on data already on the GPU: lagged covariances, k-means,
assignment to centers, transition counts, distance features, the TICA
projection and the captured moments + assignment sequence.

listed()            the cases
draw(rng)           one more case of the same ranges
prepare(case, seed) inputs, centers, models and plans
run(state)          one pass through the public entry points, with its outputs
work(case)          bytes and operations that one pass cannot do without
exact(case, seed)   the outputs in 64 bits from plain torch (None where there are none)

The inputs are made here from the seed, with torch alone.
"""
import math

import numpy as np
import torch

from pyemma_amd import dtraj
from pyemma_amd.batch import BatchedDiscretizer
from pyemma_amd.coordinates import assign_to_centers, cluster_kmeans, covariance_lagged, featurizer
from pyemma_amd.coordinates._data import DeviceTrajectories
from pyemma_amd.coordinates.koopman import KoopmanWeights
from pyemma_amd.coordinates.tica import TICA


def listed():
    return [
        # TICA's covariances of one 30-dimensional trajectory of 100,000 frames: an ordinary small system
        dict(name="cov_small", kind="cov", n=100_000, d=30, ntraj=1, lag=10, ragged=False, reversible=True,
             ctt=False, weighted=False, precision="bf16x4-acc", data="tics"),
        # TICA's covariances of the 300 pair distances of 25 particles, 200 trajectories of 50,000 frames
        dict(name="cov_features", kind="cov", n=10_000_000, d=300, ntraj=200, lag=20, ragged=False, reversible=True,
             ctt=False, weighted=False, precision="bf16x4-acc", data="distances"),
        # the covariances behind VAMP (separate means, C00, C0t and Ctt) in its default precision, ragged trajectories
        dict(name="vamp_fp64", kind="cov", n=1_500_000, d=131, ntraj=40, lag=5, ragged=True, reversible=False,
             ctt=True, weighted=False, precision="fp64", data="tics"),
        # reweighted TICA: the weighted covariances with a linear (Koopman) weight model
        dict(name="cov_weighted", kind="cov", n=2_000_000, d=150, ntraj=60, lag=10, ragged=True, reversible=True,
             ctt=False, weighted=True, precision="bf16x4-acc", data="tics"),
        # a data set of many uneven trajectories in one captured launch sequence: moments and assignment
        dict(name="batched_ragged", kind="batch", n=8_000_000, d=128, ntraj=400, lag=5, k=512, data="tics"),
        # one short trajectory against a resident center set: latency
        dict(name="assign_small", kind="assign", n=1500, d=5, k=100, ntraj=1, lag=0, data="tics"),
        # TICA-projected frames to an MSM's microstates, and the transition counts of the labels
        dict(name="discretize_tica", kind="assign", n=10_000_000, d=32, k=1000, ntraj=200, lag=20, data="tics"),
        # 10^7 frames of 300 distances to 1000 centers
        dict(name="assign_features", kind="assign", n=10_000_000, d=300, k=1000, ntraj=200, lag=0, data="distances"),
        # wide features, many centers
        dict(name="assign_wide", kind="assign", n=2_000_000, d=512, k=4096, ntraj=1, lag=0, data="mixture"),
        # k-means (kmeans++ and ten Lloyd iterations) on a TICA projection
        dict(name="kmeans_tica", kind="kmeans", n=250_000, d=10, k=200, ntraj=5, max_iter=10, data="tics"),
        # k-means on a subsample of distance features
        dict(name="kmeans_features", kind="kmeans", n=200_000, d=300, k=1000, ntraj=20, max_iter=5, data="distances"),
        # particle coordinates to pair distances to TICA components
        dict(name="features_to_tics", kind="project", n=4_000_000, atoms=25, m=10),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["cov", "cov", "batch", "assign", "assign", "assign", "kmeans", "project"])
    data = rng.choice(["tics", "distances", "mixture"])
    ntraj = _log_int(rng, 1, 400)
    if kind == "cov":
        d = _log_int(rng, 2, 300)
        reversible = rng.random() < 0.6
        weighted = rng.random() < 0.25
        precision = "fp64" if rng.random() < 0.3 else "bf16x4-acc"
        top = 3.0e11 if precision == "fp64" else 9.0e11  # n d^2
        n = _log_int(rng, 20_000, min(10_000_000, top / (d * d)))
        ntraj = min(ntraj, max(1, n // 2000))
        return dict(kind="cov", n=n, d=d, ntraj=ntraj, lag=rng.randint(1, 100), ragged=rng.random() < 0.7,
                    reversible=reversible, ctt=not reversible and not weighted, weighted=weighted,
                    precision=precision, data=data)
    if kind == "batch":
        d = _log_int(rng, 16, 200)
        n = _log_int(rng, 100_000, min(8_000_000, 1.0e9 / d))
        return dict(kind="batch", n=n, d=d, ntraj=min(ntraj, max(1, n // 2000)), lag=rng.randint(1, 50),
                    k=_log_int(rng, 32, 512), data=data)
    if kind == "assign":
        d = _log_int(rng, 2, 512)
        k = _log_int(rng, 10, 4096)
        n = _log_int(rng, 500, max(1000, min(10_000_000, 3.0e9 / d, 3.0e12 / (d * k))))
        return dict(kind="assign", n=n, d=d, k=k, ntraj=min(ntraj, max(1, n // 500)),
                    lag=rng.choice([0, 0, rng.randint(1, 100)]) if k <= 1024 else 0, data=data)
    if kind == "kmeans":
        d = _log_int(rng, 2, 300)
        k = _log_int(rng, 20, 1000)
        n = _log_int(rng, 20_000, min(250_000, 6.0e7 / d))
        return dict(kind="kmeans", n=n, d=d, k=k, ntraj=min(ntraj, max(1, n // 2000)), max_iter=rng.randint(2, 10),
                    data=data)
    atoms = rng.randint(4, 40)
    pairs = atoms * (atoms - 1) // 2
    return dict(kind="project", n=_log_int(rng, 10_000, min(4_000_000, 1.2e9 / pairs)), atoms=atoms,
                m=rng.randint(1, min(32, pairs)))


# ----------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _smooth(n, c, g, sigma):
    """(n, c) bounded, time-correlated processes: sines of diffusing phases (block by block of rows)."""
    out = torch.empty((n, c), dtype=torch.float32, device="cuda")
    phase = 2.0 * math.pi * torch.rand((1, c), generator=g, device="cuda", dtype=torch.float64)
    blk = 1 << 18
    for lo in range(0, n, blk):
        m = min(blk, n - lo)
        p = torch.randn((m, c), generator=g, device="cuda", dtype=torch.float32).mul_(sigma).to(torch.float64)
        p = phase + torch.cumsum(p, dim=0)
        phase = p[-1:].clone()
        out[lo:lo + m] = torch.sin(p).to(torch.float32)
    return out


def _positions(n, atoms, g):
    """Particles that wander around one of three basins each."""
    basins = 1.5 * torch.randn((3, 3), generator=g, device="cuda")
    home = basins[torch.randint(0, 3, (atoms,), generator=g, device="cuda")].reshape(1, 3 * atoms)
    return _smooth(n, 3 * atoms, g, 0.05).mul_(0.7).add_(home).reshape(n, atoms, 3)


def _frames(case, seed):
    """(n, d) float32 frames of the case's kind of data."""
    g = _gen(seed)
    n, d = case["n"], case["d"]
    if case["data"] == "distances":
        # distances of random pairs among as many particles as d needs (25 particles have 300 pairs)
        atoms = max(3, int(math.ceil((1.0 + math.sqrt(1.0 + 8.0 * d)) / 2.0)))
        iu, ju = np.triu_indices(atoms, k=1)
        iu, ju = torch.as_tensor(iu[:d], device="cuda"), torch.as_tensor(ju[:d], device="cuda")
        xyz = _positions(n, atoms, g)
        X = torch.empty((n, d), dtype=torch.float32, device="cuda")
        blk = 1 << 17
        for lo in range(0, n, blk):
            p = xyz[lo:lo + blk]
            X[lo:lo + blk] = (p[:, iu, :] - p[:, ju, :]).norm(dim=-1)
        return X
    if case["data"] == "mixture":
        # 64 Gaussians with anisotropic variances
        mu = 2.0 * torch.randn((64, d), generator=g, device="cuda")
        sd = torch.exp(0.5 * (math.log(0.1) + math.log(20.0) * torch.rand((64, d), generator=g, device="cuda")))
        X = torch.empty((n, d), dtype=torch.float32, device="cuda")
        blk = 1 << 19
        for lo in range(0, n, blk):
            m = min(blk, n - lo)
            c = torch.randint(0, 64, (m,), generator=g, device="cuda")
            X[lo:lo + m] = mu[c] + sd[c] * torch.randn((m, d), generator=g, device="cuda")
        return X
    # slow coordinates mixed into d columns of decreasing scale, with noise and an offset
    slow = min(d, 16)
    mix = torch.randn((slow, d), generator=g, device="cuda") / math.sqrt(slow)
    scale = 3.0 * torch.exp(-1.5 * torch.arange(d, device="cuda") / d)
    offset = 2.0 * torch.randn((1, d), generator=g, device="cuda")
    X = _smooth(n, slow, g, 0.03) @ mix
    blk = 1 << 20
    for lo in range(0, n, blk):
        m = min(blk, n - lo)
        X[lo:lo + m] += 0.3 * torch.randn((m, d), generator=g, device="cuda")
        X[lo:lo + m] *= scale
        X[lo:lo + m] += offset
    return X


def _offsets(case, seed):
    n, nt = case["n"], case["ntraj"]
    if nt == 1:
        return np.array([0, n], dtype=np.int64)
    if not case.get("ragged", case["kind"] == "batch"):
        return (np.arange(nt + 1, dtype=np.int64) * n) // nt
    # lengths log-uniform over a factor of 200
    w = np.exp(np.random.default_rng(seed).uniform(0.0, math.log(200.0), size=nt))
    cut = np.floor(np.cumsum(w) / w.sum() * n).astype(np.int64)
    cut[-1] = n
    return np.concatenate([[0], cut])


def _centers(X, k, seed):
    """k centers: means of eight consecutive frames at random places."""
    n = X.shape[0]
    g = _gen(seed + 1)
    span = min(8, n)
    at = torch.randint(0, n - span + 1, (k,), generator=g, device="cuda")
    C = torch.zeros((k, X.shape[1]), dtype=torch.float32, device="cuda")
    for i in range(span):
        C += X[at + i]
    return (C / span).cpu().numpy()


def _koopman_u(d, seed):
    """A weight model close to one with a small linear part."""
    rng = np.random.default_rng(seed + 2)
    return rng.normal(size=d) * (0.02 / math.sqrt(d)), 1.0


def _tica_model(case, seed):
    """Mean and, in the eigenbasis Q, C00 = Q s Q^T and C0t = Q s lam Q^T of a fitted TICA of all pair distances."""
    d = case["atoms"] * (case["atoms"] - 1) // 2
    rng = np.random.default_rng(seed + 3)
    Q, _ = np.linalg.qr(rng.normal(size=(d, d)))
    s = np.exp(-3.0 * np.arange(d) / d)
    lam = 0.999 * np.exp(-4.0 * np.arange(d) / d)
    return 1.0 + rng.random(d), Q, s, lam


def _tica(case, seed):
    t = TICA(lag=10, dim=case["m"])
    mean, Q, s, lam = _tica_model(case, seed)
    sym = lambda M: 0.5 * (M + M.T)
    t.model.update_model_params(mean=mean, cov=sym((Q * s) @ Q.T), cov_tau=sym((Q * (s * lam)) @ Q.T))
    t.eigenvectors  # diagonalized once, as after a fit
    return t


def prepare(case, seed):
    kind = case["kind"]
    if kind == "project":
        f = featurizer(case["atoms"])
        f.add_distances(f.pairs(np.arange(case["atoms"])))
        xyz = _positions(case["n"], case["atoms"], _gen(seed)).contiguous()
        return dict(case=case, xyz=xyz, featurizer=f, tica=_tica(case, seed))
    X = _frames(case, seed)
    offsets = _offsets(case, seed)
    if kind == "batch":
        C = _centers(X, case["k"], seed)
        return dict(case=case, plan=BatchedDiscretizer(X, offsets, case["lag"], C).capture())
    state = dict(case=case, data=DeviceTrajectories(X, offsets))
    if kind == "cov":
        state["weights"] = KoopmanWeights(*_koopman_u(case["d"], seed)) if case["weighted"] else "empirical"
    elif kind == "assign":
        state["assigner"] = assign_to_centers(centers=_centers(X, case["k"], seed))
    return state


# ----------------------------------------------------------------------
# one pass
# ----------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "cov":
        c = covariance_lagged(state["data"], c00=True, c0t=True, ctt=case["ctt"], remove_data_mean=True,
                              reversible=case["reversible"], bessel=False, lag=case["lag"],
                              weights=state["weights"], precision=case["precision"])
        out = dict(mean=c.mean, C00=c.C00_, C0t=c.C0t_)
        if case["ctt"]:
            out["Ctt"] = c.Ctt_
        return out
    if kind == "batch":
        plan = state["plan"]
        plan.replay()
        w, sx, sy, Mxx, Mxy, _ = plan.out
        return dict(w=w, sx=sx, Mxx=Mxx, Mxy=Mxy, labels=plan.labels)
    if kind == "assign":
        labels = state["assigner"].assign_device(state["data"])
        if case["lag"] == 0:
            return dict(labels=labels.S)
        return dict(labels=labels.S, counts=dtraj.count_matrix(labels, case["lag"], sparse_return=False,
                                                               nstates=case["k"]))
    if kind == "kmeans":
        km = cluster_kmeans(state["data"], k=case["k"], max_iter=case["max_iter"], fixed_seed=17)
        return dict(first=km.initial_centers_, centers=km.clustercenters, inertias=km.inertias)
    feats = state["featurizer"].transform_device(state["xyz"])
    data = DeviceTrajectories(feats, np.array([0, case["n"]], dtype=np.int64))
    return dict(features=feats, tics=state["tica"].transform_device(data))


# ----------------------------------------------------------------------
# what a pass cannot do without
# ----------------------------------------------------------------------
def _moments_work(n, d, reversible, ctt, weighted):
    # symmetric matrices count one triangle; reversible moments are two symmetric matrices
    flops = 2.0 * n * d * (d + 1) if reversible else n * d * (d + 1) * (2.0 if ctt else 1.0) + 2.0 * n * d * d
    mats = 2 + (1 if ctt else 0)
    return 4.0 * n * d + 8.0 * mats * d * d, flops + (2.0 * n * d if weighted else 0.0)


def work(case):
    n, kind = case["n"], case["kind"]
    if kind == "project":
        p = case["atoms"] * (case["atoms"] - 1) // 2
        m = case["m"]
        return dict(bytes=12.0 * n * case["atoms"] + 4.0 * n * (p + m), flops=9.0 * n * p + 2.0 * n * p * m)
    d = case["d"]
    if kind == "cov":
        b, f = _moments_work(n, d, case["reversible"], case["ctt"], case["weighted"])
        return dict(bytes=b, flops=f)
    k = case["k"]
    if kind == "batch":
        b, f = _moments_work(n, d, True, False, False)
        return dict(bytes=b + 4.0 * n + 4.0 * k * d, flops=f + 2.0 * n * k * d)
    if kind == "assign":
        return dict(bytes=4.0 * n * d + 4.0 * n + 4.0 * k * d + (8.0 * k * k if case["lag"] else 0.0),
                    flops=2.0 * n * k * d)
    # k - 1 rounds of distances to one center, then max_iter assignments to k centers
    return dict(bytes=4.0 * n * d + 8.0 * k * d, flops=3.0 * n * d * (k - 1) + 2.0 * n * k * d * case["max_iter"])


# ----------------------------------------------------------------------
# 64-bit values
# ----------------------------------------------------------------------
def _exact_moments(X, offsets, lag, reversible, u=None):
    """(w, sx, sy, Cxx, Cxy, Cyy): FP64 sums and mean-free comoments over all pairs (row, row + lag)."""
    d = X.shape[1]
    z = dict(dtype=torch.float64, device="cuda")
    w = 0.0
    sx, sy = torch.zeros(d, **z), torch.zeros(d, **z)
    xx, xy, yy = torch.zeros((d, d), **z), torch.zeros((d, d), **z), torch.zeros((d, d), **z)
    shift = X[:: max(1, X.shape[0] // 64)].double().mean(dim=0)
    for t in range(len(offsets) - 1):
        a, b = int(offsets[t]), int(offsets[t + 1]) - lag
        for lo in range(a, b, 1 << 20):
            hi = min(b, lo + (1 << 20))
            x, y = X[lo:hi].double() - shift, X[lo + lag:hi + lag].double() - shift
            if u is None:
                wt, wx, wy = float(hi - lo), x, y
            else:
                q = X[lo:hi].double() @ torch.as_tensor(u[0], **z) + u[1]
                wt, wx, wy = float(q.sum()), x * q[:, None], y * q[:, None]
            w += wt
            sx += wx.sum(dim=0)
            sy += wy.sum(dim=0)
            xx += wx.T @ x
            xy += wx.T @ y
            yy += wy.T @ y
    if reversible:
        w, sx = 2.0 * w, sx + sy
        sy, xx, xy = sx, xx + yy, xy + xy.T
        yy = xx
    xx = xx - torch.outer(sx, sx) / w
    xy = xy - torch.outer(sx, sy) / w
    yy = yy - torch.outer(sy, sy) / w
    return w, sx + w * shift, sy + w * shift, xx, xy, yy


def exact(case, seed):
    kind = case["kind"]
    if kind == "cov":
        X, offsets = _frames(case, seed), _offsets(case, seed)
        u = _koopman_u(case["d"], seed) if case["weighted"] else None
        w, sx, sy, xx, xy, yy = _exact_moments(X, offsets, case["lag"], case["reversible"], u)
        h = lambda t: (t / w).cpu().numpy()
        out = dict(mean=h(sx), C00=h(xx), C0t=h(xy))
        if case["ctt"]:
            out["Ctt"] = h(yy)
        return out
    if kind == "batch":
        X, offsets = _frames(case, seed), _offsets(case, seed)
        w, sx, sy, xx, xy, _ = _exact_moments(X, offsets, case["lag"], True)
        return dict(w=torch.tensor([w], dtype=torch.float64, device="cuda"), sx=sx, Mxx=xx, Mxy=xy, labels=None)
    if kind == "project":
        atoms, n = case["atoms"], case["n"]
        xyz = _positions(n, atoms, _gen(seed))
        iu, ju = np.triu_indices(atoms, k=1)
        iu, ju = torch.as_tensor(iu, device="cuda"), torch.as_tensor(ju, device="cuda")
        feats = torch.empty((n, len(iu)), dtype=torch.float64, device="cuda")
        blk = 1 << 17
        for lo in range(0, n, blk):
            p = xyz[lo:lo + blk].double()
            feats[lo:lo + blk] = (p[:, iu, :] - p[:, ju, :]).norm(dim=-1)
        # the kinetic map's eigenvectors, each with its largest element positive
        mean, Q, s, lam = _tica_model(case, seed)
        V = Q[:, :case["m"]] / np.sqrt(s[:case["m"]])
        V = V * np.sign(V[np.argmax(np.abs(V), axis=0), np.arange(V.shape[1])]) * lam[:case["m"]]
        mean, V = torch.as_tensor(mean, device="cuda"), torch.as_tensor(V, device="cuda")
        tics = torch.empty((n, case["m"]), dtype=torch.float64, device="cuda")
        for lo in range(0, n, blk):
            tics[lo:lo + blk] = (feats[lo:lo + blk].float().double() - mean) @ V
        return dict(features=feats, tics=tics)
    return None  # labels and cluster centers are chosen, not computed
