"""Sponge runs on models whose tiles lie inside the undamped part (no strip, no
top row), below and on both sides of the rule that picks the rows per wavefront
(70, 511 and 512 tiles): receivers, strided snapshots and the previous level
against the FP64 oracle, forward and in reverse, at the tolerance of the other
sponge tests (FP32 against FP64, relative L2 1e-5), and the same bit for bit in
pieces of one, two and several steps."""
import numpy as np
import pytest

import oracle
import sssi_amd
from sssi_amd import synth

pytestmark = pytest.mark.gpu

SIZES = [(150, 300, 10), (112, 3504, 12), (256, 1536, 9)]
NT, DT, STRIDE = 48, 1e-3, 5


def _model(nz, nx):
    rng = np.random.default_rng(nz + nx)
    return np.asfortranarray(1500.0 + 2000.0 * rng.random((nz, nx)))


def _near(a, b):
    return np.linalg.norm(a - b) <= 1e-5 * np.linalg.norm(b)


@pytest.mark.parametrize("nz, nx, nB", SIZES)
def test_forward(nz, nx, nB):
    v = _model(nz, nx)
    w = synth.ricker(40.0, NT, DT)
    iz, ix = [0, nz // 2, nz // 2, nz - 1], [nx // 2, nx // 3, nx // 3 + 1, 3]
    ww = np.stack([w * (1 + 0.5 * k) for k in range(4)], axis=1)
    print(f"sponge forward {nz}x{nx} nB={nB}", flush=True)
    d, s = sssi_amd.fwd_sponge_2d_points(v, NT, nB, 10.0, 10.0, DT, iz, ix, ww,
                                         want_snapshot=True, snap_stride=STRIDE)
    do, so = oracle.fwd_sponge_2d(v, NT, nB, 10.0, 10.0, DT, src_iz=iz, src_ix=ix, wavelet=ww,
                                  want_snapshot=True, snap_stride=STRIDE)
    assert _near(d, do)
    for k in range(1, s.shape[2]):
        assert _near(s[:, :, k], so[:, :, k]), k
    for pieces in ([1] * NT, [2] * (NT // 2), [1, 2, 8, 3, 34]):
        p = sssi_amd.Propagator(v, 1, nB, 10.0, 10.0, DT, abc="sponge")
        p.set_points(iz, ix, ww)
        t = 0
        for n in pieces:
            p.run_steps(t, n)
            t += n
            if (t - 1) % STRIDE == 0:
                assert np.array_equal(p.field(), s[:, :, (t - 1) // STRIDE]), (pieces, t)
        assert np.array_equal(p.data(NT), d), pieces


@pytest.mark.parametrize("nz, nx, nB", SIZES)
def test_reverse(nz, nx, nB):
    v = _model(nz, nx)
    data = np.asfortranarray(np.random.default_rng(nx).standard_normal((nx, NT)))
    print(f"sponge reverse {nz}x{nx} nB={nB}", flush=True)
    m, s = sssi_amd.rvs_sponge_2d_ex(v, data, nB, 10.0, 10.0, DT, snap_stride=STRIDE)
    mo, so = oracle.rvs_sponge_2d(v, data, nB, 10.0, 10.0, DT, want_snapshot=True,
                                  snap_stride=STRIDE)
    assert _near(m, mo)
    for k in range(s.shape[2]):
        assert _near(s[:, :, k], so[:, :, k]), k
    for pieces in ([1] * NT, [2] * (NT // 2), [1, 2, 8, 3, 34]):
        p = sssi_amd.Propagator(v, 1, nB, 10.0, 10.0, DT, abc="sponge")
        p.set_surface(data)
        t = NT - 1
        for n in pieces:
            p.run_steps(t, n, reverse=True)
            t -= n
        assert np.array_equal(p.model(), m) and np.array_equal(p.field(), s[:, :, 0]), pieces
