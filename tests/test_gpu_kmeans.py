"""GPU kmeans++ and Lloyd through the C ABI vs the C oracle (identical picks,
bit-identical centers, inertias and labels)."""
import numpy as np
import pytest

from oracle import native as on
from pyemma_amd import _native

pytestmark = pytest.mark.gpu


def _kmpp(X, k, seed):
    t = _native.torch()
    C, idx = _native.kmeanspp(_native.as_device_f32(X), k, seed)
    t.cuda.synchronize()
    return C.cpu().numpy(), idx.cpu().numpy()


def _lloyd(X, C0, max_iter, tol, mode):
    t = _native.torch()
    Xt = _native.as_device_f32(X)
    C = _native.as_device_f32(C0).clone()
    labels, inert, n_iter, conv = _native.lloyd(Xt, C, max_iter, tol, mode=mode)
    t.cuda.synchronize()
    it = int(n_iter.item())
    return C.cpu().numpy(), labels.cpu().numpy(), inert.cpu().numpy()[:it], bool(conv.item())


@pytest.mark.parametrize("n,d,k,seed", [(9000, 3, 6, 1), (20000, 30, 50, 42), (5000, 300, 20, 7),
                                        (4097, 2, 300, 3), (100, 4, 100, 9)])
def test_kmeanspp_identical_picks(n, d, k, seed):
    rng = np.random.default_rng(seed)
    X = (rng.standard_normal((n, d)) * rng.uniform(0.5, 2, d)).astype(np.float32)
    C_ref, idx_ref = on.kmeanspp(X, k, seed, nthreads=4)
    C, idx = _kmpp(X, k, seed)
    np.testing.assert_array_equal(idx, idx_ref)
    np.testing.assert_array_equal(C, C_ref)


@pytest.mark.parametrize("n,d,k,scale,shift", [
    (5000, 7, 40, 1.0, 0), (8193, 64, 33, 1.0, 0), (8193, 64, 33, 1.0, 1), (5000, 131, 40, 1.0, 0),
    (3000, 126, 20, 1.0, 1), (3000, 63, 20, 1.0, 0), (3000, 60, 20, 1.0, 1), (4096, 4, 130, 1.0, 0), (1, 3, 3, 1.0, 0),
    (270000, 3, 12, 1.0, 0), (300, 16384, 5, 1.0, 0), (4097, 20, 30, 1e-14, 0), (4097, 20, 30, 1e-20, 0),
    (4097, 20, 30, 1e19, 0), (4097, 20, 30, 1e25, 0)])
def test_kmeanspp_skipped_frames(n, d, k, scale, shift):
    """Separated groups, so that the triangle inequality leaves out most frames of a
    round: picks identical at block and superblock edges, in rows that are not 16-byte
    aligned, and where distances underflow or overflow (no frame may be left out)."""
    t = _native.torch()
    rng = np.random.default_rng(n + d)
    X = (rng.standard_normal((n, d)) + 40.0 * rng.standard_normal((9, d))[rng.integers(0, 9, n)])
    X = (X * scale).astype(np.float32)
    with np.errstate(over="ignore"):
        C_ref, idx_ref = on.kmeanspp(X, k, 3, nthreads=4)
    buf = t.empty(n * d + shift, dtype=t.float32, device="cuda")
    Xt = buf[shift:].view(n, d)
    Xt.copy_(t.from_numpy(X))
    C, idx = _native.kmeanspp(Xt, k, 3)
    np.testing.assert_array_equal(idx.cpu().numpy(), idx_ref)
    np.testing.assert_array_equal(C.cpu().numpy(), C_ref)


def test_kmeanspp_duplicate_points_total_zero():
    X = np.repeat(np.arange(3, dtype=np.float32)[:, None], 50, axis=0)
    C_ref, idx_ref = on.kmeanspp(X, 5, 11)
    C, idx = _kmpp(X, 5, 11)
    np.testing.assert_array_equal(idx, idx_ref)


@pytest.mark.parametrize("mode", [_native.EMMA_ASSIGN_FP32_PLAIN, _native.EMMA_ASSIGN_BF16X3_RECHECK])
@pytest.mark.parametrize("n,d,k", [(6000, 5, 12), (9000, 30, 100), (3000, 300, 40)])
def test_lloyd_bit_identical(mode, n, d, k):
    rng = np.random.default_rng(n + k)
    X = (rng.standard_normal((n, d)) + rng.integers(0, 4, (n, 1)) * 3.0).astype(np.float32)
    C0, _ = on.kmeanspp(X, k, 5)
    C_ref, lab_ref, in_ref, conv_ref = on.lloyd(X, C0, 8, 0.0, nthreads=4)
    C, lab, inert, conv = _lloyd(X, C0, 8, 0.0, mode)
    np.testing.assert_array_equal(inert, in_ref)
    np.testing.assert_array_equal(C, C_ref)
    np.testing.assert_array_equal(lab, lab_ref)
    assert conv == conv_ref


def test_lloyd_converges_and_stops(golden_hmm):
    g = golden_hmm
    C, lab, inert, conv = _lloyd(g["X"], g["kmpp_centers"], 5, 0.0, _native.EMMA_ASSIGN_BF16X3_RECHECK)
    np.testing.assert_array_equal(C, g["lloyd_centers"])
    np.testing.assert_array_equal(inert, g["lloyd_inertias"])
    X = np.zeros((40000, 4), dtype=np.float32)
    for i, v in enumerate([30.0, 60.0, 90.0, 120.0]):
        X[i * 10000:(i + 1) * 10000] = v
    C0, _ = on.kmeanspp(X, 4, 42)
    C, lab, inert, conv = _lloyd(X, C0, 10, 1e-5, _native.EMMA_ASSIGN_BF16X3_RECHECK)
    assert sorted(C[:, 0].tolist()) == [30.0, 60.0, 90.0, 120.0]
    assert conv and len(inert) < 10


@pytest.mark.parametrize("n,d,k", [(1, 3, 1), (4097, 3, 1), (63, 2, 5), (4096, 4, 64), (8200, 3, 1024), (9000, 2, 1025),
                                   (70000, 2, 2100)])
def test_lloyd_member_order_edges(n, d, k):
    """Label counts, offsets and the stable member order at the edges of a group of 64
    frames, a block of 4096, 16 blocks and 1024 labels: bit-identical means and costs."""
    rng = np.random.default_rng(n + k)
    X = rng.standard_normal((n, d)).astype(np.float32)
    C0 = X[rng.permutation(n)[:k]].copy()
    C_ref, lab_ref, in_ref, _ = on.lloyd(X, C0, 3, 0.0, nthreads=4)
    C, lab, inert, _ = _lloyd(X, C0, 3, 0.0, _native.EMMA_ASSIGN_BF16X3_RECHECK)
    np.testing.assert_array_equal(lab, lab_ref)
    np.testing.assert_array_equal(inert, in_ref)
    np.testing.assert_array_equal(C, C_ref)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("d", list(range(1, 24)) + [31, 32, 33, 47, 48, 63])
def test_kmeanspp_row_remainders(d, shift):
    """Rows of every length around the 16 dims that are read together, aligned and not."""
    t = _native.torch()
    rng = np.random.default_rng(d)
    n = 700
    X = (rng.standard_normal((n, d)) + 3.0 * rng.standard_normal((6, d))[rng.integers(0, 6, n)]).astype(np.float32)
    C_ref, idx_ref = on.kmeanspp(X, 25, 4, nthreads=4)
    buf = t.empty(n * d + shift, dtype=t.float32, device="cuda")
    Xt = buf[shift:].view(n, d)
    Xt.copy_(t.from_numpy(X))
    C, idx = _native.kmeanspp(Xt, 25, 4)
    np.testing.assert_array_equal(idx.cpu().numpy(), idx_ref)
    np.testing.assert_array_equal(C.cpu().numpy(), C_ref)


@pytest.mark.parametrize("n,d,k,shift", [(65_536, 64, 6, 0), (65_537, 64, 6, 0), (6_103, 8192, 4, 0), (6_104, 8192, 4, 0),
                                         (70, 8192, 20, 1), (70, 8193, 20, 0), (900, 301, 30, 1), (300, 1000, 30, 0)])
def test_kmeanspp_own_or_staged_rows(n, d, k, shift):
    """Both ways of reading rows of 64 dims and more, on either side of each line."""
    t = _native.torch()
    rng = np.random.default_rng(n + d)
    X = rng.standard_normal((n, d), dtype=np.float32)
    X += 3.0 * rng.standard_normal((6, d), dtype=np.float32)[rng.integers(0, 6, n)]
    C_ref, idx_ref = on.kmeanspp(X, k, 4, nthreads=8)
    buf = t.empty(n * d + shift, dtype=t.float32, device="cuda")
    Xt = buf[shift:].view(n, d)
    Xt.copy_(t.from_numpy(X))
    C, idx = _native.kmeanspp(Xt, k, 4)
    np.testing.assert_array_equal(idx.cpu().numpy(), idx_ref)
    np.testing.assert_array_equal(C.cpu().numpy(), C_ref)
