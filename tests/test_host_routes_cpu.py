"""Which kernels a call launches, without a GPU: the choice between two forms
of a kernel where the wrong one gives the same values more slowly."""
import pytest

import hipmock

_HELM = """
from sssi_amd import helmholtz
m = np.full(({nz}, {nx}), 2000.0 ** -2, order="F")
S = np.zeros(({nz} * {nx}, 1), dtype=np.complex128)
helmholtz.solve(m, S, 60.0, {N}, 1, 10.0, 10.0)
for k in ("freq_lu", "freq_subst", "freq_panel", "freq_trail_lds", "freq_trail", "freq_solve"):
    print(k, count(k))
"""


def _helm(nz, nx, N, before="", **env):
    out = hipmock.run(before + _HELM.format(nz=nz, nx=nx, N=N), **env)
    n = {k: int(v) for k, v in (line.split() for line in out.splitlines())}
    n["freq_trail"] -= n["freq_trail_lds"]  # (counted by part of the name)
    return {k for k, v in n.items() if v}


BLOCKED = {"freq_lu", "freq_subst"}
REPLAY = {"freq_panel", "freq_trail_lds", "freq_solve"}
GLOBAL = {"freq_panel", "freq_trail", "freq_solve"}


@pytest.mark.parametrize("nz, nx, N, form", [
    (40, 10, 1, BLOCKED), (160, 4, 2, BLOCKED),                # bands 40, 480
    (161, 4, 2, REPLAY), (300, 4, 2, REPLAY),                  # 483, 900
    (332, 4, 2, REPLAY), (336, 4, 2, REPLAY),                  # 996, 1008: 1024 rows
    (337, 4, 2, GLOBAL),                                       # 1011
    (200, 5, 3, REPLAY), (128, 8, 5, REPLAY),                  # 1000, 1152 in 1000, 1024 unknowns
])
def test_helmholtz_form(nz, nx, N, form):
    """Rows of a panel in 512 threads' registers, else in 1024 LDS rows, else
    in global memory."""
    assert _helm(nz, nx, N) == form


@pytest.mark.parametrize("nc", ["1", "2", "4"])
def test_helmholtz_replay_on_request(nc):
    assert _helm(40, 10, 1, SSSI_FREQ_NC=nc) == REPLAY


@pytest.mark.parametrize("free, form", [(1 << 38, BLOCKED), (1_300_000_000, REPLAY)])
def test_helmholtz_panels_that_do_not_fit(free, form):
    """1.1 GB of panels (band 40, 1.2e6 unknowns) with and without the room for
    them: without, the form that needs none."""
    n = _helm(40, 30000, 1, before=f"M.hipmock_mem_free({free})\n")
    assert n == form


_SPONGE = """
v = np.full(({nz}, {nx}), 2000.0, order="F")
P = sssi_amd.Propagator(v, 1, 5, 10.0, 10.0, 1e-3, abc="sponge")
P.set_points([0], [1], np.zeros(64))
M.hipmock_clear()
P.run_steps(0, {n})
print(count("sponge2d_stepILi"), count("sponge2d_steps"))
"""


@pytest.mark.parametrize("nz, nx, n, single, several", [
    (100, 150, 1, 1, 0), (100, 150, 2, 0, 1), (100, 150, 8, 0, 1), (100, 150, 17, 1, 2),
    (515, 1203, 1, 1, 0), (515, 1203, 2, 2, 0), (515, 1203, 3, 0, 1), (515, 1203, 10, 2, 1),
])
def test_sponge_pieces(nz, nx, n, single, several):
    """Pieces of one step, and of two on a full chip, take the one-step kernel."""
    out = hipmock.run(_SPONGE.format(nz=nz, nx=nx, n=n)).split()
    assert [int(x) for x in out] == [single, several]


_SOURCES = """
v = np.full((100, 150), 2000.0, order="F")
P = sssi_amd.Propagator(v, {N}, 5, 10.0, 10.0, 1e-3, abc="{abc}")
k = np.arange({n})
P.set_points(k // 150, k % 150, np.zeros((16, {n})))
M.hipmock_clear()
P.run_steps(0, 16)
print(count("steps") - count("ELb1EE"), count("ELb1EE"))
"""


@pytest.mark.parametrize("abc, N, n, few, many", [
    ("sponge", 1, 4, 2, 0), ("sponge", 1, 5, 0, 2), ("sponge", 1, 2000, 0, 2),
    ("cpml", 1, 4, 2, 0), ("cpml", 1, 5, 0, 2), ("cpml", 2, 8, 4, 0), ("cpml", 2, 9, 0, 4),
    ("cpml", 2, 64, 0, 4), ("cpml", 2, 65, 0, 0),
])
def test_sources_per_launch(abc, N, n, few, many):
    """Launches of several steps that loop over all sources, and that test 64 at
    a time; CPML with more than 64 sources takes its one-step kernel."""
    out = hipmock.run(_SOURCES.format(abc=abc, N=N, n=n)).split()
    assert [int(x) for x in out] == [few, many]


@pytest.mark.parametrize("layout", ["8x24", "4x32", "plain"])
def test_eikonal_fills_one_level(layout):
    """The first launch writes every cell of the other level."""
    out = hipmock.run("""
V = np.full((90, 70), 2000.0, order="F")
sssi_amd.eikonal2d_batch(V, 10.0, [1, 1], [3, 60], 12)
print(count("eik_init"))
""", SSSI_EIK=layout)
    assert int(out) == 1
