"""Row affine map out = X u + u0 at the edges of a wave's rows and columns, and the weight
sums of trajectories around a workgroup's batches of loads."""
import numpy as np
import pytest

from pyemma_amd import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 9, 31, 32, 33, 1001])
@pytest.mark.parametrize("d", [1, 63, 64, 65, 150])
def test_row_affine(n, d):
    rng = np.random.default_rng(n * d)
    X = rng.standard_normal((n, d)).astype(np.float32)
    u = rng.standard_normal(d)
    out = _native.row_affine(_native.as_device_f32(X), u, 0.5).cpu().numpy()
    # d products and sums in FP64, each within 2^-53 of the sum of the magnitudes
    bound = (d + 8) * 2.0 ** -53 * (np.abs(X.astype(np.float64)) @ np.abs(u) + 0.5)
    assert np.all(np.abs(out - (X.astype(np.float64) @ u + 0.5)) <= bound)


@pytest.mark.parametrize("pairs", [1, 255, 4095, 4096, 4097, 8448, 20000])
def test_weight_sums(pairs):
    t = _native.torch()
    rng = np.random.default_rng(pairs)
    n = pairs + 3
    X = rng.standard_normal((n, 5)).astype(np.float32)
    wts = rng.random(n) + 0.5
    w = _native.moments_lagged(_native.as_device_f32(X), np.array([0, n]), 3, reversible=True,
                               precision=_native.EMMA_PREC_FP64, weights=t.from_numpy(wts).cuda())[0]
    ref = wts[:pairs].sum()
    assert abs(float(w.item()) - 2 * ref) <= 2 * ref * pairs * 2.0 ** -53 or abs(float(w.item()) - ref) <= ref * pairs * 2.0 ** -53


@pytest.mark.parametrize("pairs", [1, 255, 4095, 4096, 4097, 8448, 20000])
@pytest.mark.parametrize("stride", [1, 3])
@pytest.mark.parametrize("precision", ["fp64", "bf16x4-acc"])
def test_weighted_moments(pairs, stride, precision):
    """Reversible weighted moments around the batches of the weight sums: the total, the sums
    and both matrices, so that every pair's weight counts."""
    from pyemma_amd.coordinates.covariance import PRECISIONS

    t = _native.torch()
    rng = np.random.default_rng(pairs + stride)
    lens = [3 + (pairs - 1) * stride + 1, 3 + 40 * stride]  # the second one: 40 pairs
    n = sum(lens)
    X = (rng.standard_normal((n, 5)) + 0.3).astype(np.float32)
    wts = rng.random(n) + 0.5
    off = np.array([0, lens[0], n])
    w, sx, _, Mxx, Mxy, _ = _native.moments_lagged(_native.as_device_f32(X), off, 3, stride=stride, reversible=True,
                                                   precision=PRECISIONS[precision], weights=t.from_numpy(wts).cuda())
    at = np.concatenate([np.arange(a, b - 3, stride) for a, b in zip(off[:-1], off[1:])])
    assert len(at) == pairs + 40
    q, x, y = wts[at], X[at].astype(np.float64), X[at + 3].astype(np.float64)
    rw, rs = 2 * q.sum(), q @ (x + y)
    A = (x * q[:, None]).T @ y
    rxx = (x * q[:, None]).T @ x + (y * q[:, None]).T @ y - np.outer(rs, rs) / rw
    rxy = A + A.T - np.outer(rs, rs) / rw
    # magnitudes of the summed products around any shift within the data's range
    m = np.abs(X).max() + np.abs(x) + np.abs(y)
    big = 2 * (m * q[:, None]).T @ m
    u = 2.0 ** -53 * (len(at) + 16)
    # two operands to 2^-17, their sums over 64 products and the weights to FP32
    e = u if precision == "fp64" else 2 * 2.0 ** -17 + 66 * 2.0 ** -24
    f = u if precision == "fp64" else u + 4 * 2.0 ** -24
    assert abs(float(w.item()) - rw) <= u * rw
    assert np.all(np.abs(sx.cpu().numpy() - rs) <= f * 2 * (q @ m))
    assert np.all(np.abs(Mxx.cpu().numpy() - rxx) <= e * big)
    assert np.all(np.abs(Mxy.cpu().numpy() - rxy) <= e * big)


@pytest.mark.parametrize("n,d", [(16383, 400), (16384, 400), (16389, 400), (50_000, 100), (50_001, 100), (20_000, 3)])
def test_row_affine_many_rows(n, d):
    """Either side of the sizes from which a wave takes eight rows: the same sums."""
    rng = np.random.default_rng(n + d)
    X = rng.standard_normal((n, d)).astype(np.float32)
    u = rng.standard_normal(d)
    out = _native.row_affine(_native.as_device_f32(X), u, 0.5).cpu().numpy()
    bound = (d + 8) * 2.0 ** -53 * (np.abs(X.astype(np.float64)) @ np.abs(u) + 0.5)
    assert np.all(np.abs(out - (X.astype(np.float64) @ u + 0.5)) <= bound)
    parts = [_native.row_affine(_native.as_device_f32(X[a:a + 1000]), u, 0.5).cpu().numpy() for a in range(0, n, 1000)]
    np.testing.assert_array_equal(out, np.concatenate(parts))
