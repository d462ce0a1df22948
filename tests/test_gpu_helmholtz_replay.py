"""Column-replay factorisation against the oracle, bit for bit: one, two and
four rows per thread (systems of up to 256, 512 and 1024 rows), the panel in
global memory (more than 636 rows), the replay in global memory (more than 1024
rows), and one, two and four columns per workgroup, with column counts that are
no multiple of it."""
import numpy as np
import pytest

import oracle
from sssi_amd import helmholtz

pytestmark = pytest.mark.gpu

CASES = [  # nz, nx, N, nB, f               band, unknowns
    (61, 4, 5, 2, 30.0),    # 549, 244
    (61, 8, 5, 2, 30.0),    # 549, 488
    (161, 5, 2, 2, 25.0),   # 483, 805
    (131, 7, 3, 2, 20.0),   # 655, 917
    (336, 4, 2, 1, 20.0),   # 1008, 1344
    (351, 4, 2, 1, 20.0),   # 1053, 1404
]


def _match(nz, nx, N, nB, f):
    rng = np.random.default_rng(nz + nx)
    m = np.asfortranarray(1.0 / (1500.0 + 2500.0 * rng.random((nz, nx))) ** 2)
    w, n = 2 * np.pi * f, nz * nx
    S = np.zeros((n, 2), dtype=np.complex128)
    S[n // 2, 0] = 1.0
    S[:, 1] = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    U = helmholtz.solve(m, S, w, N, nB, 10.0, 12.5)
    assert np.array_equal(U, oracle.freq_cpml_2d_solve(m, S, w, N, nB, 10.0, 12.5))


@pytest.mark.parametrize("nc", ["", "1", "4"])
@pytest.mark.parametrize("nz, nx, N, nB, f", CASES)
def test_replay_matches_oracle(nz, nx, N, nB, f, nc, monkeypatch):
    if nc:
        monkeypatch.setenv("SSSI_FREQ_NC", nc)
    print(f"helmholtz replay {nz}x{nx} N={N} nc={nc}", flush=True)
    _match(nz, nx, N, nB, f)


@pytest.mark.parametrize("nz, nx, N, nB, f", [(37, 23, 1, 3, 25.0), (41, 9, 2, 2, 30.0)])
def test_trailing_columns_in_part_groups(nz, nx, N, nB, f):
    """Blocked form: column counts behind the panel that are no multiple of the
    workgroup's four (851 and 369 unknowns), a reach that ends inside a group."""
    print(f"helmholtz blocked {nz}x{nx} N={N}", flush=True)
    _match(nz, nx, N, nB, f)
