"""Kirchhoff migration at the edges of its index arithmetic and of its two
forms: sample indices near both ends of 32 bits are refused as any other outside
the record, and calls whose grids of patches, images or traces are beyond the
grouped form's limits take the other one (SSSI_KIRCH=stack by name), with the
same stack and images bit for bit."""
import numpy as np
import pytest

import hipmock
import sssi_amd
from sssi_amd import kirchhoff

DT = 2e-3


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["", "stack"])
@pytest.mark.parametrize("ks, kr", [
    (-2147483000, -2147483290), (-2147483648, -2147482000), (2147483647, 2147483647),
    (-5, 3), (2147483647, -5)])
def test_indices_outside_the_record(ks, kr, form, monkeypatch):
    """Their 32-bit sum may wrap round into the record (the first gives 1006)."""
    monkeypatch.setenv("SSSI_KIRCH", form)
    nz, nx, nt = 3, 4, 2000
    T = np.zeros((nz, nx, 2), order="F")
    T[:, :, 0], T[:, :, 1] = (ks - 1) * DT, (kr - 1) * DT
    shot = np.asfortranarray(np.random.default_rng(1).standard_normal((nt, nx)))
    print(f"kirchhoff indices {ks} {kr} {form}", flush=True)
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


@pytest.mark.gpu
@pytest.mark.parametrize("shots", [1, 4, 5, 7])
@pytest.mark.parametrize("images", [False, True])
def test_stack_form(shots, images, monkeypatch):
    rng = np.random.default_rng(shots)
    V = np.asfortranarray(np.sort(1500.0 + 1500.0 * rng.random((37, 50)), axis=0))
    xsr = np.arange(1, 51, 3)
    K = kirchhoff.Kirchhoff2D(V, 10.0, xsr, 45, DT)
    K.load_shots(rng.standard_normal((900, 50, shots)))
    ixs = rng.choice(np.arange(1, xsr.size + 1), shots, replace=False)
    print(f"kirchhoff stack {shots} images={images}", flush=True)
    a = K.migrate_loaded(xsr, ixs, images=images)
    monkeypatch.setenv("SSSI_KIRCH", "stack")
    b = K.migrate_loaded(xsr, ixs, images=images)
    for p, q in zip(a if images else [a], b if images else [b]):
        assert np.array_equal(p, q) and np.any(p != 0)


_WIDE = """
import sssi_amd._lib as L
M.hipmock_copy_limit(1 << 20)
nx = {nx}
T = np.zeros((1, nx, 1), order="F")
shot = np.zeros((1, nx), order="F")
m = np.zeros((1, nx), order="F")
one = np.array([1], dtype=np.int32)
rc = sssi_amd.lib().sssi_kirchhoff_migrate(L._dp(T), 1, nx, 1, L._ip(one), 1, L._ip(one), 1,
                                           L._dp(shot), 1, 1e-3, 1, L._dp(m))
print(rc, count("kirch_group"), count("kirch_stack"))
"""


@pytest.mark.parametrize("nx, group", [(1 << 27, 1), (1 << 28, 0)])
def test_more_patches_than_a_grid_holds(nx, group):
    """One row of 2^28 columns is 2^26 patches of 64 threads, a thread more than
    a launch takes."""
    assert hipmock.run(_WIDE.format(nx=nx)).split() == ["0", str(group), str(1 - group)]
