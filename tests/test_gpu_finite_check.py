"""Non-finite input is refused wherever the value stands, also where the check rides on
the results of the call (column sums, undecided frames, projections), and finite input
whose sums or distances overflow is not."""
import numpy as np
import pytest

from pyemma_amd import _native
from pyemma_amd.coordinates.clustering import AssignCenters
from pyemma_amd.coordinates.covariance import LaggedCovariance
from pyemma_amd.coordinates.tica import TICA
from pyemma_amd.exceptions import InvalidDataInStreamException

pytestmark = pytest.mark.gpu
BAD = [np.nan, np.inf, -np.inf]


@pytest.mark.parametrize("d", [1, 31, 32, 130, 300, 512])
@pytest.mark.parametrize("n,k", [(5, 1), (5, 40), (300, 2), (3000, 1), (3000, 70), (40000, 33)])
def test_assignment(n, k, d):
    rng = np.random.default_rng(n + k + d)
    X = rng.standard_normal((n, d)).astype(np.float32)
    C = rng.standard_normal((k, d)).astype(np.float32)
    cl = AssignCenters(C)
    ref = cl.assign(X)
    before = cl.n_rechecked
    for i, bad in enumerate(BAD + BAD):
        Y = X.copy()
        Y[(0, n - 1, int(rng.integers(n)))[i % 3], int(rng.integers(d))] = bad
        with pytest.raises(InvalidDataInStreamException):
            cl.assign(Y)
        with pytest.raises(InvalidDataInStreamException):
            cl.assign_device(Y)
        assert cl.n_rechecked == before
    Y = X.copy()
    Y[n // 2] = 3e38
    plain = AssignCenters(C, assign_mode="fp32")
    np.testing.assert_array_equal(cl.assign(Y), plain.assign(Y))
    np.testing.assert_array_equal(cl.assign(X), ref)
    with pytest.raises(ValueError):
        cl.assign(np.ones((4, d + 1), np.float32))


@pytest.mark.parametrize("opts", [
    dict(lag=3), dict(lag=0, c0t=False), dict(lag=3, reversible=True), dict(lag=3, ctt=True),
    dict(lag=3, reversible=True, precision="fp64"), dict(lag=3, ctt=True, precision="fp64"),
    dict(lag=3, reversible=True, remove_data_mean=True), dict(lag=60, reversible=True), dict(lag=3, stride=2),
    dict(lag=3, skip=5, reversible=True), dict(lag=3, c0t=False), dict(lag=3, weights=2.0)])
@pytest.mark.parametrize("d", [1, 20, 65, 131, 300])
def test_covariances(opts, d):
    rng = np.random.default_rng(d)
    opts = dict(dict(c00=True, c0t=True), **opts)
    lens = [400, 101, 5000]
    X = [rng.standard_normal((T, d)).astype(np.float32) for T in lens]
    cov = LaggedCovariance(**opts)
    cov.partial_fit(X)
    C00 = cov.C00_
    for i, bad in enumerate(BAD + BAD):
        Y = [x.copy() for x in X]
        # the first and last rows; with lag 60, a row of the second trajectory that is in no pair
        j, row = [(0, 0), (2, 4999), (1, 50)][i % 3]
        Y[j][row, int(rng.integers(d))] = bad
        with pytest.raises(InvalidDataInStreamException):
            cov.partial_fit(Y)
        with pytest.raises(InvalidDataInStreamException):
            LaggedCovariance(**opts).estimate(Y)
        np.testing.assert_array_equal(cov.C00_, C00)
    Y = [x.copy() for x in X]
    Y[2][17:900:6] = 3e38  # finite: accepted
    LaggedCovariance(**opts).estimate(Y)


@pytest.mark.parametrize("d,m", [(2, 1), (33, 5), (300, 10)])
def test_projection(d, m):
    rng = np.random.default_rng(d)
    X = np.cumsum(rng.standard_normal((2000, d)), axis=0).astype(np.float32)
    tica = TICA(lag=2, dim=m)
    tica.estimate(X)
    Y0 = tica.transform(X)
    for i, bad in enumerate(BAD + BAD):
        Y = X.copy()
        Y[(0, 1999, 777)[i % 3], int(rng.integers(d))] = bad
        for call in (tica.transform, tica.transform_device, TICA(lag=2, dim=m).estimate):
            with pytest.raises(InvalidDataInStreamException):
                call(Y)
    with pytest.raises(InvalidDataInStreamException):
        TICA(lag=2, dim=d + 1).estimate(Y)
    np.testing.assert_array_equal(tica.transform(X), Y0)
    Y = X.copy()
    Y[5] = 3e38
    assert tica.transform(Y).shape == (2000, m)


@pytest.mark.parametrize("shift", [0, 1, 2, 3])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 7, 8, 63, 1029, 40007])
def test_count_at_every_alignment(n, shift):
    t = _native.torch()
    buf = t.full((n + shift + 8,), float("nan"), device="cuda")
    x = buf[shift:shift + n]
    x.zero_()
    assert int(_native.count_nonfinite(x).item()) == 0
    where = sorted({0, n // 2, max(n - 4, 0), n - 1})
    for i, w in enumerate(where):
        x[w] = BAD[i % 3]
        assert int(_native.count_nonfinite(x).item()) == i + 1


@pytest.mark.parametrize("row", [0, 299])
@pytest.mark.parametrize("bad", BAD)
def test_rows_of_no_trajectory(row, bad):
    """A device matrix with rows in front of the first trajectory or behind the last is
    refused for what they hold too."""
    from pyemma_amd.coordinates._data import DeviceTrajectories
    from pyemma_amd.coordinates.vamp import VAMP

    t = _native.torch()
    X = t.randn((300, 4), generator=t.Generator(device="cuda").manual_seed(2), device="cuda")
    dt = DeviceTrajectories(X, np.array([10, 150, 280]))
    calls = [LaggedCovariance(c00=True, c0t=True, lag=3).estimate, TICA(lag=3, dim=2).estimate,
             VAMP(lag=3, dim=2).estimate]
    for call in calls:
        call(dt)
    X[row, 1] = bad
    for call in calls:
        with pytest.raises(InvalidDataInStreamException):
            call(dt)
