"""Batched uneven trajectories in one captured launch sequence (the config-4 shape, reduced).

96 linear-Langevin trajectories with log-uniform lengths 200 - 6,000 frames,
d = 128, lag 5, k = 512 centers: the eager pass matches the FP64 oracle
(moments) and the sequential FP32 oracle (labels); every graph replay, with
eager work and synchronizations in between, reproduces the eager results
bit for bit, also after new frames are copied into the captured input.
"""
import numpy as np
import pytest

from oracle import moments as om
from oracle import native as on
from pyemma_amd import _native, autotune
from pyemma_amd.batch import BatchedDiscretizer
from pyemma_amd.synthetic import langevin_trajectories

pytestmark = pytest.mark.gpu


def _close(a, b, rtol=2e-5, atol_rel=1e-5):
    np.testing.assert_allclose(a, b, rtol=rtol, atol=atol_rel * np.abs(b).max())


def test_batched_graph_replay_matches_eager_and_oracle():
    t = _native.torch()
    X, off = langevin_trajectories(96, 128, lmin=200, lmax=6000, seed=4)
    Xh = X.cpu().numpy()
    trajs = [Xh[a:b] for a, b in zip(off[:-1], off[1:])]
    rng = np.random.default_rng(0)
    C = Xh[np.sort(rng.choice(len(Xh), 512, replace=False))].copy()
    b = BatchedDiscretizer(X, off, 5, C)
    w, mean, C00, C0t, labels = b.run_eager()
    ref = om.covariance_lagged(trajs, 5, remove_data_mean=True, reversible=True, bessel=False)
    assert w == ref["w"]
    _close(mean, ref["mean"], rtol=1e-6)
    _close(C00, ref["C00"])
    _close(C0t, ref["C0t"])
    assert np.array_equal(labels, on.assign(Xh, C, nthreads=8))
    assert autotune.tuned(), "autotuner did not run"

    b.capture()
    for i in range(3):
        b.replay()
        t.cuda.synchronize()
        r = b.results()
        assert r[0] == w
        for x, y in zip(r[1:], (mean, C00, C0t, labels)):
            assert np.array_equal(x, y), "replay %d differs from the eager pass" % i
        # eager work of the program between replays
        _native.assign(b.X[:1000], b.C)
        t.cuda.synchronize()

    # new frames into the captured input: replay == eager on the new data
    X2, _ = langevin_trajectories(96, 128, lmin=200, lmax=6000, seed=5,
                                  lengths=np.diff(off))
    b.X.copy_(X2)
    b.replay()
    t.cuda.synchronize()
    r = b.results()
    e = BatchedDiscretizer(X2, off, 5, C).run_eager()
    assert r[0] == e[0]
    for x, y in zip(r[1:], e[1:]):
        assert np.array_equal(x, y)


def test_replay_after_larger_calls():
    """Larger assignment and moments calls after the capture replace the shared scratch
    buffers: the replays still give the eager results and write into no other tensor."""
    t = _native.torch()
    X, off = langevin_trajectories(12, 40, lmin=200, lmax=900, seed=8)
    C = X[::37].cpu().numpy()[:60].copy()
    b = BatchedDiscretizer(X, off, 5, C)
    ref = b.run_eager()
    b.capture()
    g = t.Generator(device="cuda").manual_seed(1)
    big = t.randn((300_000, 40), generator=g, device="cuda")
    _native.assign(big, big[:500].contiguous())
    _native.moments_lagged(big, np.array([0, len(big)]), 5, precision=_native.EMMA_PREC_BF16X4_ACC)
    t.cuda.synchronize()
    # tensors of many sizes, over whatever the calls above gave back
    others = [t.full((1 << p,), 17, dtype=t.uint8, device="cuda") for p in range(12, 26) for _ in range(4)]
    for i in range(3):
        b.labels.fill_(-5)
        b.replay()
        t.cuda.synchronize()
        r = b.results()
        assert r[0] == ref[0]
        for x, y in zip(r[1:], ref[1:]):
            assert np.array_equal(x, y), "replay %d" % i
        assert all(bool((o == 17).all()) for o in others), "replay %d wrote into another tensor" % i
        _native.assign(big[:1000], big[:500].contiguous())


def test_results_are_those_of_the_last_pass():
    """results() after capture() are the warm-up's, after a replay the replay's, also where
    an eager pass ran in between."""
    t = _native.torch()
    X, off = langevin_trajectories(5, 9, lmin=300, lmax=700, seed=3)
    X2 = (X * 1.5 + 0.25).contiguous()
    C = X[::50].cpu().numpy().copy()
    b = BatchedDiscretizer(X.clone(), off, 4, C)

    def same(r, ref):
        return all(np.array_equal(x, y) for x, y in zip(r, ref))

    ref = BatchedDiscretizer(X, off, 4, C).run_eager()
    ref2 = BatchedDiscretizer(X2, off, 4, C).run_eager()
    b.capture()
    assert same(b.results(), ref)
    held = b.out  # every replay writes these
    for _ in range(2):
        b.X.copy_(X2)
        assert same(b.run_eager(), ref2)
        b.X.copy_(X)
        b.replay()
        t.cuda.synchronize()
        assert same(b.results(), ref)
        assert b.out is held
