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
