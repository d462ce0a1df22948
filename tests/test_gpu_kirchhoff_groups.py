"""Kirchhoff migration's shot groups against the oracle, bit for bit: every
group size (1 to 8 shots, and counts that split into equal groups), images at
and around the wave's 16 x 4 patch, receiver counts that are no multiple of the
receivers in flight, and an index past the record at each group size."""
import numpy as np
import pytest

import oracle
import sssi_amd

pytestmark = pytest.mark.gpu


def _case(nz, nx, nshot, nt, seed):
    rng = np.random.default_rng(seed)
    V = np.asfortranarray(1500.0 + 50.0 * np.arange(nz)[:, None] + 20.0 * rng.random((nz, nx)))
    xsr = np.arange(1, nx + 1)
    shots = rng.standard_normal((nt, nx, nshot))
    return V, xsr, shots, rng.integers(1, nx + 1, nshot)


@pytest.mark.parametrize("nshot", [1, 2, 3, 4, 5, 6, 7, 8, 9, 17])
@pytest.mark.parametrize("nz, nx", [(16, 4), (15, 9), (33, 21)])
def test_groups_match_oracle(nz, nx, nshot):
    dt, nt = 1e-3, 900
    V, xsr, shots, ixs = _case(nz, nx, nshot, nt, 10 * nshot + nx)
    print(f"kirchhoff groups {nz}x{nx} shots={nshot}", flush=True)
    k = sssi_amd.Kirchhoff2D(V, 10.0, xsr, nz + nx, dt)
    tt = k.travel_time()
    for xrec in (xsr, xsr[1::2], xsr[:1]):
        stack, images = k.migrate_shots(xrec, shots, ixs, images=True)
        ref = np.zeros((nz, nx))
        for s in range(nshot):
            M = oracle.kirchhoff_migrate(tt, xrec, xsr, shots[:, :, s], dt, nz, int(ixs[s]))
            assert np.array_equal(images[:, :, s], M)
            ref = ref + M
        assert np.array_equal(stack, ref)
    # no receivers: zero images
    assert not k.migrate_shots(np.zeros(0, dtype=int), shots, ixs).any()
    with pytest.raises(sssi_amd.SssiError):
        k.migrate_shots(xsr, shots[:3], ixs)
    k.close()
