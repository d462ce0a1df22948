"""Results that come to the host in pinned chunks with worker threads (more
than one chunk of 8 MB, one chunk, less than a worker's share, concurrent
calls) and snapshots turned to z-fastest on the device: equal to the same
values fetched in small pieces or computed without snapshots."""
import threading

import numpy as np
import pytest

import oracle
import sssi_amd
from sssi_amd import synth

pytestmark = pytest.mark.gpu


def _model(nz, nx, seed):
    rng = np.random.default_rng(seed)
    return np.asfortranarray(1500.0 + 1500.0 * rng.random((nz, nx)))


@pytest.mark.parametrize("n", [1, 2, 90])  # 0.1, 0.2, 9.4 MB of tables
def test_tables_over_chunks(n):
    V = _model(117, 112, 1)
    sx = 1 + np.arange(n) % 112
    print(f"downloads {n} tables", flush=True)
    T = sssi_amd.eikonal2d_batch(V, 10.0, np.ones(n, dtype=int), sx, 40)
    for k in {0, n // 2, n - 1}:
        assert np.array_equal(T[:, :, k], sssi_amd.eikonal2d(V, 10.0, 1, int(sx[k]), 40))


def test_concurrent_calls():
    V = _model(64, 200, 2)
    ref = sssi_amd.eikonal2d_batch(V, 10.0, np.ones(200, dtype=int), np.arange(1, 201), 20)
    out = [None] * 4

    def run(k):
        out[k] = sssi_amd.eikonal2d_batch(V, 10.0, np.ones(200, dtype=int), np.arange(1, 201), 20)
    th = [threading.Thread(target=run, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for o in out:
        assert np.array_equal(o, ref)


@pytest.mark.parametrize("nz, nx", [(63, 64), (65, 130), (129, 63)])
def test_snapshots_2d(nz, nx):
    v, nt, dt = _model(nz, nx, nz), 40, 1e-3
    w = synth.ricker(30, nt, dt)
    d, s = sssi_amd.fwd_cpml_2d_points(v, nt, 2, 5, 10.0, 10.0, dt, [0], [nx // 2], w,
                                       want_snapshot=True, snap_stride=1)
    p = sssi_amd.Propagator(v, 2, 5, 10.0, 10.0, dt)
    p.set_points([0], [nx // 2], w)
    t = 0
    for n in (1, 12, 27):
        p.run_steps(t, n)
        t += n
        assert np.array_equal(p.field(), s[:, :, t - 1])
    assert np.array_equal(p.data(nt), d)


def test_snapshots_3d():
    rng = np.random.default_rng(3)
    v = np.asfortranarray(1500.0 + 800.0 * rng.random((33, 70, 21)))
    nt, dt = 12, 1e-3
    w = synth.ricker(40, nt, dt)
    args = (v, nt, 2, 4, 10.0, 10.0, 10.0, dt)
    d, s = sssi_amd.fwd_cpml_3d_points(*args, [1], [35], [9], w, want_snapshot=True, snap_stride=5)
    p = sssi_amd.Propagator(v, 2, 4, 10.0, 10.0, dt, dy=10.0)
    p.set_points([1], [35], w, src_iy=[9])
    p.run_steps(0, 11)
    assert np.array_equal(p.field(), s[:, :, :, 2])
    ref, rs = oracle.fwd_cpml_3d(*args, src_iz=[1], src_ix=[35], src_iy=[9], wavelet=w,
                                 want_snapshot=True, snap_stride=5)
    assert np.linalg.norm(s - rs) <= 1e-5 * np.linalg.norm(rs)
