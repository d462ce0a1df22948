"""Work lists of the blocked eikonal passes (a launch runs only the tiles whose
input can have changed) against the oracle, bit for bit: grids at and around
the tile centre's size (56 x 24 at the default layout), models in which a front
comes back to tiles that had settled (a fast channel under slow ground), pass
counts that stop a front midway, and more tiles than a launch has blocks."""
import numpy as np
import pytest

import oracle
import sssi_amd

pytestmark = pytest.mark.gpu


def _channel(nz, nx, seed):
    """Slow ground with a fast floor and a slow block: late, repeated updates."""
    rng = np.random.default_rng(seed)
    V = 400.0 + 200.0 * rng.random((nz, nx))
    V[2 * nz // 3:, :] = 5000.0
    V[nz // 4:nz // 2, nx // 3:nx // 2] = 30.0
    return np.asfortranarray(V)


@pytest.mark.parametrize("nz, nx", [(2, 2), (56, 24), (57, 25), (112, 48), (113, 97), (170, 61)])
@pytest.mark.parametrize("frac", [0.1, 0.6, 1.5])
def test_lists_match_oracle(nz, nx, frac):
    V = _channel(nz, nx, nz + nx)
    iMax = max(1, int(frac * (nz + nx) / 4))
    sz, sx = [1, nz, nz // 2 + 1], [1, nx, nx // 2 + 1]
    print(f"eikonal lists {nz}x{nx} iMax={iMax}", flush=True)
    T = sssi_amd.eikonal2d_batch(V, 10.0, sz, sx, iMax)
    for k in range(3):
        assert np.array_equal(T[:, :, k], oracle.eikonal2d(V, 10.0, sz[k], sx[k], iMax))


def test_more_tiles_than_blocks():
    nz, nx, n = 60, 50, 700  # 2 x 3 tiles per table
    V = _channel(nz, nx, 4)
    rng = np.random.default_rng(1)
    sz, sx = rng.integers(1, nz + 1, n), rng.integers(1, nx + 1, n)
    print("eikonal lists, 4200 tiles", flush=True)
    T = sssi_amd.eikonal2d_batch(V, 10.0, sz, sx, 45)
    for k in range(0, n, 37):
        assert np.array_equal(T[:, :, k], oracle.eikonal2d(V, 10.0, int(sz[k]), int(sx[k]), 45))
