"""Narrow tiles (8 passes per launch on 64 x 24) of small eikonal calls: grids at and
around the written part of a tile (48 x 8), pass counts that are no multiple of 8,
and tables on both sides of the rule's line (3e6 cells), bit for bit against the
oracle and against the wide tiles (SSSI_EIK=4x32)."""
import numpy as np
import pytest

import oracle
import sssi_amd

pytestmark = pytest.mark.gpu


def _model(nz, nx):
    rng = np.random.default_rng(nz * 3 + nx)
    V = 400.0 + 200.0 * rng.random((nz, nx))
    V[2 * nz // 3:, :] = 5000.0
    return np.asfortranarray(V)


@pytest.mark.parametrize("nz, nx", [(2, 3), (47, 8), (48, 9), (49, 7), (97, 17), (144, 64)])
@pytest.mark.parametrize("iMax", [1, 3, 26, 61])
def test_narrow_tiles_match_oracle(monkeypatch, nz, nx, iMax):
    V, sz, sx = _model(nz, nx), [1, nz, nz // 2 + 1], [nx, 1, nx // 2 + 1]
    print(f"eikonal narrow {nz}x{nx} iMax={iMax}", flush=True)
    T = sssi_amd.eikonal2d_batch(V, 10.0, sz, sx, iMax)
    for k in range(3):
        assert np.array_equal(T[:, :, k], oracle.eikonal2d(V, 10.0, sz[k], sx[k], iMax))
    monkeypatch.setenv("SSSI_EIK", "4x32")
    assert np.array_equal(T, sssi_amd.eikonal2d_batch(V, 10.0, sz, sx, iMax))


@pytest.mark.parametrize("n", [12, 13])  # 500 x 500: 3.0e6 and 3.25e6 cells
def test_both_sides_of_the_line(monkeypatch, n):
    V, s = _model(500, 500), list(range(1, 500, 38))[:n]
    print(f"eikonal narrow, {n} tables", flush=True)
    T = sssi_amd.eikonal2d_batch(V, 10.0, [1] * n, s, 150)
    for layout in ("4x32", "8x24"):
        monkeypatch.setenv("SSSI_EIK", layout)
        assert np.array_equal(T, sssi_amd.eikonal2d_batch(V, 10.0, [1] * n, s, 150))
