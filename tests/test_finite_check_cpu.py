"""Which trajectories the column sums of a moments call take in completely, so that they
can stand for the check of the input for non-finite values."""
import numpy as np
import pytest
import torch

from pyemma_amd.coordinates._data import DeviceTrajectories
from pyemma_amd.coordinates.covariance import LaggedCovariance


@pytest.mark.parametrize("offsets,covered", [
    ([0, 100], True), ([0, 40, 100], True), ([0, 6, 100], True), ([0, 5, 100], False), ([0, 3, 100], False),
    ([0, 90], False), ([0, 40, 99], False), ([1, 100], False), ([10, 40, 90], False)])
def test_rows_outside_the_sums(offsets, covered):
    dt = DeviceTrajectories(torch.zeros((100, 3)), np.array(offsets))
    assert bool(LaggedCovariance(c00=True, c0t=True, lag=3)._sums_cover(dt)) is covered
