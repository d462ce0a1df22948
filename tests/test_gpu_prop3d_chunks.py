"""The z chunk of a 3-D grid by its size: on grids on both sides of the rule's
lines (384 and 640 blocks of 32 planes) and of less than a chunk, the layout is
the rule's, and receivers and field equal those of 32- and 20-plane chunks bit for
bit (a cell's arithmetic does not depend on the chunk it lies in)."""
import numpy as np
import pytest

import sssi_amd
from sssi_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N, nz, nx, ny, nB, zc", [
    (2, 5, 9, 11, 0, 8), (4, 33, 70, 30, 6, 8), (1, 384, 64, 256, 10, 8), (3, 385, 64, 256, 10, 24),
    (4, 320, 128, 256, 12, 24), (2, 321, 128, 256, 12, 32)])
def test_chunk_rule(monkeypatch, N, nz, nx, ny, nB, zc):
    rng = np.random.default_rng(nz)
    v, nt, dt = 1500.0 + 2000.0 * rng.random((nz, nx, ny)), 14, 5e-4
    iz, ix, iy = [1, nz - 1], [nx // 2, nx // 3], [ny // 2, ny - 2]
    ww = np.stack([synth.ricker(30, nt, dt)] * 2, axis=1)
    print(f"3-D chunks N={N} {nz}x{nx}x{ny} nB={nB}", flush=True)

    def run():
        p = sssi_amd.Propagator(v, N, nB, 10.0, 10.0, dt, dy=10.0)
        p.set_points(iz, ix, ww, iy)
        p.run(nt)
        return p.layout(), p.data(nt), p.field()
    rule = run()
    assert rule[0] == (8, zc) and np.abs(rule[2]).max() > 0
    for z in ("32", "20"):
        monkeypatch.setenv("SSSI_ZC3", z)
        lay, d, f = run()
        assert lay[1] == int(z) and np.array_equal(d, rule[1]) and np.array_equal(f, rule[2])
