"""Kirchhoff migration at the edges of its index arithmetic: sample indices near
both ends of 32 bits are refused as any other outside the record."""
import numpy as np
import pytest

import sssi_amd
from sssi_amd import kirchhoff

DT = 2e-3


@pytest.mark.gpu
@pytest.mark.parametrize("ks, kr", [
    (-2147483000, -2147483290), (-2147483648, -2147482000), (2147483647, 2147483647),
    (-5, 3), (2147483647, -5)])
def test_indices_outside_the_record(ks, kr):
    """Their 32-bit sum may wrap round into the record (the first gives 1006)."""
    nz, nx, nt = 3, 4, 2000
    T = np.zeros((nz, nx, 2), order="F")
    T[:, :, 0], T[:, :, 1] = (ks - 1) * DT, (kr - 1) * DT
    shot = np.asfortranarray(np.random.default_rng(1).standard_normal((nt, nx)))
    print(f"kirchhoff indices {ks} {kr}", flush=True)
    with pytest.raises(sssi_amd.SssiError) as e:
        kirchhoff.migrate(T, [2], [1, 2], shot, DT, nz, 1)
    assert e.value.code == -1


@pytest.mark.gpu
def test_indices_at_the_ends_that_meet_inside():
    """A strongly negative and a strongly positive index whose sum is a sample."""
    nz, nx, nt = 3, 4, 2000
    T = np.zeros((nz, nx, 2), order="F")
    T[:, :, 0], T[:, :, 1] = (-2147483000 - 1) * DT, (2147483640 - 1) * DT
    shot = np.asfortranarray(np.random.default_rng(1).standard_normal((nt, nx)))
    m = kirchhoff.migrate(T, [2], [1, 2], shot, DT, nz, 1)
    assert np.array_equal(m, np.full((nz, nx), shot[639, 1]))
