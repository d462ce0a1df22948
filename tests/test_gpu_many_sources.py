"""Launches of several steps with few and many point sources (up to the
line between the two ways to find them, one register of 64, its edges, several), coincident ones among them, wavelets that end before
the run does: equal bit for bit to the same steps one at a time, and to the
FP64 oracle at the tolerance of the other tests (relative L2 1e-5)."""
import numpy as np
import pytest

import oracle
import sssi_amd
from sssi_amd import synth

pytestmark = pytest.mark.gpu

NZ, NX, NT, NW, DT = 70, 110, 40, 31, 1e-3


def _sources(n):
    rng = np.random.default_rng(n)
    idx = rng.choice(NZ * NX, n, replace=False)
    idx[n // 2:n // 2 + n // 8] = idx[:n // 8]  # coincident
    if n >= 16:
        idx[-8:] = 5 * NX + 60 + np.arange(8)   # side by side
    w = synth.ricker(45.0, NW, DT)[:, None] * rng.uniform(0.5, 2.0, n)
    return idx // NX, idx % NX, np.ascontiguousarray(w)


@pytest.mark.parametrize("n", [1, 4, 5, 8, 9, 63, 64, 65, 129, 1500])
@pytest.mark.parametrize("abc, N", [("sponge", 1), ("cpml", 1), ("cpml", 2), ("cpml", 3), ("cpml", 4)])
def test_sources(abc, N, n):
    rng = np.random.default_rng(3)
    v = np.asfortranarray(1500.0 + 1500.0 * rng.random((NZ, NX)))
    iz, ix, w = _sources(n)
    print(f"sources {abc} N={N} n={n}", flush=True)

    def run(pieces):
        p = sssi_amd.Propagator(v, N, 9, 10.0, 10.0, DT, abc=abc)
        p.set_points(iz, ix, w)
        t = 0
        for k in pieces:
            p.run_steps(t, k)
            t += k
        return p.data(NT), p.field()
    d, f = run([NT])
    for pieces in ([1] * NT, [7, 33]):
        a, b = run(pieces)
        assert np.array_equal(a, d) and np.array_equal(b, f), pieces
    # the wavefield, not the receivers: few deep sources reach those with values
    # below FP32's normal range only
    full = np.zeros((NT, n))
    full[:NW] = w
    kw = dict(src_iz=iz, src_ix=ix, wavelet=full, want_snapshot=True, snap_stride=NT - 1)
    if abc == "sponge":
        _, s = oracle.fwd_sponge_2d(v, NT, 9, 10.0, 10.0, DT, **kw)
    else:
        _, s = oracle.fwd_cpml_2d(v, NT, N, 9, 10.0, 10.0, DT, **kw)
    o = s[:, :, 1]
    assert np.linalg.norm(f - o) <= 1e-5 * np.linalg.norm(o)
