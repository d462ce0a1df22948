"""Several 2-D CPML steps per launch: receivers, field, previous level and
snapshots equal those of one step per launch (SSSI_STEPS=0) bit for bit, forward
and in reverse, whole and in uneven pieces with single steps between, on models
at and around the written part of a tile (N=1 16 x 48, 2 8 x 40, 3 18 x 34,
4 4 x 36), smaller than its rim, without strips and with strips that meet, and
on both sides of the tile counts and the source count (64) that the several-step
launch ends at."""
import numpy as np
import pytest

import sssi_amd
from sssi_amd import synth

pytestmark = pytest.mark.gpu

# N, nz, nx, nB
CASES = [(1, 16, 48, 3), (1, 17, 97, 8), (1, 50, 130, 0), (1, 511, 1536, 20), (1, 513, 1537, 20),
         (2, 8, 40, 4), (2, 9, 41, 0), (2, 65, 193, 31), (2, 320, 640, 20), (2, 321, 641, 20),
         (3, 18, 34, 6), (3, 55, 103, 11), (3, 288, 544, 20), (3, 289, 545, 20),
         (4, 7, 9, 2), (4, 31, 73, 15), (4, 64, 576, 12), (4, 65, 577, 12), (5, 40, 90, 10)]


def _model(nz, nx):
    rng = np.random.default_rng(nz * 7 + nx)
    return np.asfortranarray(1500.0 + 2000.0 * rng.random((nz, nx)))


def _sources(nz, nx, nt, dt, n):
    rng = np.random.default_rng(n)
    iz, ix = rng.integers(0, nz, n), rng.integers(0, nx, n)
    iz[:3], ix[:3] = [0, nz - 1, nz - 1], [nx // 2, nx - 1, nx - 1]  # one cell twice
    w = synth.ricker(30, nt, dt)
    return iz, ix, np.stack([w * (1 + 0.25 * k) for k in range(n)], axis=1)


def _both(monkeypatch, run):
    monkeypatch.setenv("SSSI_STEPS", "0")
    one = run()
    monkeypatch.delenv("SSSI_STEPS")
    return one, run()


def _same(a, b, what):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert np.isfinite(x).all() and np.array_equal(x, y), what


@pytest.mark.parametrize("N, nz, nx, nB", CASES)
def test_forward(monkeypatch, N, nz, nx, nB):
    v, nt, dt = _model(nz, nx), 47, 5e-4
    print(f"cpml2d steps N={N} {nz}x{nx} nB={nB}", flush=True)
    for nsrc in (5, 64, 65):
        iz, ix, ww = _sources(nz, nx, nt, dt, nsrc)

        def run(pieces=(nt,)):
            p = sssi_amd.Propagator(v, N, nB, 10.0, 10.0, dt)
            p.set_points(iz, ix, ww)
            t = 0
            for n in pieces:
                p.run_steps(t, n)
                t += n
            return p.data(nt), p.field(), p.model()
        one, many = _both(monkeypatch, run)
        assert np.abs(one[1]).max() > 0
        _same(one, many, nsrc)
        _same(one, run((1, 2, 9, 1, 1, 33)), nsrc)

    def snaps(stride=3):
        return sssi_amd.fwd_cpml_2d_points(v, nt, N, nB, 10.0, 10.0, dt, iz, ix, ww,
                                           want_snapshot=True, snap_stride=stride)
    iz, ix, ww = _sources(nz, nx, nt, dt, 5)
    _same(*_both(monkeypatch, snaps), "snapshots")


@pytest.mark.parametrize("N, nz, nx, nB", CASES)
def test_reverse(monkeypatch, N, nz, nx, nB):
    v, nt, dt = _model(nz, nx), 38, 5e-4
    data = np.random.default_rng(2).standard_normal((nx, nt))
    print(f"cpml2d reverse steps N={N} {nz}x{nx} nB={nB}", flush=True)

    def run(pieces=(nt,)):
        p = sssi_amd.Propagator(v, N, nB, 10.0, 10.0, dt)
        p.set_surface(data)
        t = nt - 1
        for n in pieces:
            p.run_steps(t, n, reverse=True)
            t -= n
        return p.field(), p.model()
    one, many = _both(monkeypatch, run)
    _same(one, many, "reverse")
    _same(one, run((3, 1, 34)), "reverse pieces")
    _same(*_both(monkeypatch, lambda: sssi_amd.rvs_cpml_2d_ex(v, data, N, nB, 10.0, 10.0, dt,
                                                              snap_stride=5)), "reverse snapshots")
