"""Host side of the several-step 2-D CPML launches, without a GPU: a handle
whose second set of wavefields could not be allocated is as it was before the
call, and the next run allocates the whole set."""
import pytest

import hipmock

_ALLOCATION_FAILS = """
import sssi_amd._lib as L
v = np.full((60, 100), 2000.0, order="F")
P = sssi_amd.Propagator(v, 2, 10, 10.0, 10.0, 1e-3)
P.set_points([0], [50], synth.ricker(20.0, 12, 1e-3))
P.run_steps(0, 1)
class Out(ctypes.Structure):  # Steps2DOut: p, pold, zphi, zpsi, xphi, xpsi
    _fields_ = [("q", ctypes.c_void_p * 6)]
import os
M.hipmock_fail_malloc({k})
try:
    P.run_steps(1, 3, record=False)
    raise SystemExit("the run did not allocate")
except sssi_amd.SssiError as e:
    assert e.code == -2, e.code
M.hipmock_fail_malloc(-1)
M.hipmock_clear()
watch("cpml2d_steps", {job}, 48)
P.run_steps(1, 8, record=False)
n = count("cpml2d_steps")
assert n == 2, n
seen = []
for i in range(n):
    out = arg(i, 1, Out)
    assert all(out.q), (i, list(out.q))
    assert len(set(out.q)) == 6
P.field()
print("ok")
"""


@pytest.mark.parametrize("k", range(4))
def test_failed_allocation_leaves_the_handle_whole(k):
    """The k-th buffer of the second set (two levels, two memory variables) is
    refused; before it was held to be there from then on, and the next run
    wrote through its null address."""
    assert "ok" in hipmock.run(_ALLOCATION_FAILS.format(k=k, job=8))
