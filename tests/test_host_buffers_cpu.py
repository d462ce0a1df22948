"""Host side of device buffers that a handle keeps, without a GPU: one that
could not be allocated is not taken for one that is there."""
import pytest

import hipmock

_MIGRATE = """
V = np.asfortranarray(np.linspace(1500.0, 3000.0, 20)[:, None] * np.ones((1, 30)))
xsr = np.arange(1, 31)
K = sssi_amd.Kirchhoff2D(V, 10.0, xsr, 12, 2e-3)
K.load_shots(np.zeros((40, 30, 2)))
M.hipmock_fail_malloc({k})
try:
    K.migrate_loaded(xsr, [3, 7])
    raise SystemExit("the call did not allocate")
except sssi_amd.SssiError as e:
    assert e.code == -2, e.code
M.hipmock_fail_malloc(-1)
M.hipmock_clear()
# kidx, nz, nx, ntz, ts, nshot, tr, xr, nrec, shots, nt, images, bad
watch("kirch_group", 8, 4, 4, 4, 8, 4, 8, 8, 4, 8, 4, 8, 8)
K.migrate_loaded(xsr, [3, 7])
assert count("kirch_group") == 1
for a in (0, 4, 6, 7, 9, 11, 12):
    assert arg(0, a, ctypes.c_void_p).value, a
print("ok")
"""


@pytest.mark.parametrize("k", range(6))  # stack, images, shot and receiver tables, flag
def test_migration_after_a_failed_allocation(k):
    assert "ok" in hipmock.run(_MIGRATE.format(k=k))
