"""Work lists of the blocked eikonal passes at each tile layout, by name: more
tiles than a launch has blocks (2560), so that a block takes several list
entries and its LDS several tiles; grids smaller than a tile and at its edges;
against one pass per launch, bit for bit."""
import numpy as np
import pytest

import sssi_amd

pytestmark = pytest.mark.gpu

LAYOUTS = ["4x32", "4x64", "8x24", "8x48", "8x64"]


def _both(monkeypatch, layout, V, sz, sx, iMax):
    monkeypatch.setenv("SSSI_EIK", layout)
    a = sssi_amd.eikonal2d_batch(V, 10.0, sz, sx, iMax)
    monkeypatch.setenv("SSSI_EIK", "plain")
    b = sssi_amd.eikonal2d_batch(V, 10.0, sz, sx, iMax)
    return a, b


@pytest.mark.parametrize("layout", LAYOUTS)
@pytest.mark.parametrize("nz, nx, n, iMax", [
    (2, 2, 1, 3), (48, 8, 2, 20), (49, 9, 2, 20), (56, 24, 3, 25), (57, 25, 3, 25),
    (130, 190, 5, 90), (60, 50, 3, 1),
])
def test_edges(layout, nz, nx, n, iMax, monkeypatch):
    rng = np.random.default_rng(nz * nx)
    V = np.asfortranarray(1500.0 + 2500.0 * rng.random((nz, nx)))
    print(f"eikonal {layout} {nz}x{nx} n={n}", flush=True)
    a, b = _both(monkeypatch, layout, V, rng.integers(1, nz + 1, n), rng.integers(1, nx + 1, n), iMax)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("layout, n", [("4x32", 90), ("8x24", 40), ("8x48", 120)])
def test_several_tiles_per_block(layout, n, monkeypatch):
    """Tiles of 56 x 24, 48 x 8 and 48 x 32 written cells: 3360, 4480 and 2880."""
    rng = np.random.default_rng(n)
    V = np.asfortranarray(1500.0 + 2500.0 * rng.random((200, 200)))
    print(f"eikonal {layout} {n} tables", flush=True)
    a, b = _both(monkeypatch, layout, V, rng.integers(1, 201, n), rng.integers(1, 201, n), 110)
    assert np.array_equal(a, b)
