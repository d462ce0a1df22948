"""Several sponge steps per launch: one run equals the same steps run one at a
time and in uneven pieces, bit for bit (receivers, field and previous level),
forward and in reverse, on models at and around the size of a tile's written
part (16 x 48) and of the rule that picks the rows per wavefront (512 tiles);
and the forward run matches the oracle to the tolerance of the other sponge
tests (FP32 against FP64, relative L2 1e-5)."""
import numpy as np
import pytest

import oracle
import sssi_amd
from sssi_amd import synth

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 0), (16, 48, 3), (17, 49, 8), (31, 97, 0), (33, 95, 15), (263, 1490, 20),
         (250, 1553, 31)]


def _model(nz, nx):
    rng = np.random.default_rng(nz + nx)
    return np.asfortranarray(1500.0 + 2000.0 * rng.random((nz, nx)))


@pytest.mark.parametrize("nz, nx, nB", SIZES)
def test_forward_pieces_and_oracle(nz, nx, nB):
    v, nt, dt = _model(nz, nx), 61, 1e-3
    w = synth.ricker(30, nt, dt)
    iz, ix = [0, nz - 1, nz // 2, nz // 2], [nx // 2, nx - 1, nx // 3, nx // 3]
    ww = np.stack([w * (1 + 0.5 * k) for k in range(4)], axis=1)
    print(f"sponge steps {nz}x{nx} nB={nB}", flush=True)

    def run(pieces):
        p = sssi_amd.Propagator(v, 1, nB, 10.0, 10.0, dt, abc="sponge")
        p.set_points(iz, ix, ww)
        t = 0
        for n in pieces:
            p.run_steps(t, n)
            t += n
        return p.data(nt), p.field(), p.model()
    whole = run([nt])
    for pieces in ([1] * nt, [8, 16, 7, 30], [3, 5, 53]):
        for a, b in zip(whole, run(pieces)):
            assert np.array_equal(a, b), pieces
    d, _ = oracle.fwd_sponge_2d(v, nt, nB, 10.0, 10.0, dt, src_iz=iz, src_ix=ix, wavelet=ww)
    assert np.linalg.norm(whole[0] - d) <= 1e-5 * np.linalg.norm(d)


@pytest.mark.parametrize("nz, nx, nB", SIZES[1:5])
def test_reverse_pieces_and_snapshots(nz, nx, nB):
    v, nt, dt = _model(nz, nx), 43, 1e-3
    data = np.random.default_rng(2).standard_normal((nx, nt))
    print(f"sponge reverse steps {nz}x{nx} nB={nB}", flush=True)

    def run(pieces):
        p = sssi_amd.Propagator(v, 1, nB, 10.0, 10.0, dt, abc="sponge")
        p.set_surface(data)
        t = nt - 1
        for n in pieces:
            p.run_steps(t, n, reverse=True)
            t -= n
        return p.field(), p.model()
    whole = run([nt])
    for pieces in ([1] * nt, [9, 34]):
        for a, b in zip(whole, run(pieces)):
            assert np.array_equal(a, b), pieces
    m, s = sssi_amd.rvs_sponge_2d_ex(v, data, nB, 10.0, 10.0, dt, snap_stride=3)
    assert np.array_equal(m, whole[1]) and np.array_equal(s[:, :, 0], whole[0])
    for stride in (1, 5):
        _, q = sssi_amd.rvs_sponge_2d_ex(v, data, nB, 10.0, 10.0, dt, snap_stride=stride)
        for t in range(0, nt, 3 * stride):
            assert np.array_equal(q[:, :, t // stride], s[:, :, t // 3])
