"""Host side of the downloads (pinned chunks, worker threads), without a GPU:
what comes out is what is in device memory at every size around the chunk and
the worker's share, the workers do not keep the CPU busy while the GPU works,
and a host allocation that fails ends in an error code."""
import pytest

import hipmock

# (device memory of the double is host memory; the model's upload is done by a
# kernel, so fields are filled here through the handle's own record buffer)
_VALUES = """
V = np.full((8, {nx}), 2000.0, order="F")
P = sssi_amd.Propagator(V, 1, 0, 10.0, 10.0, 1e-3)
P.set_points([0], [1], np.zeros({nt}))
watch("cpml2d_steps", 1024)
P.run({nt})
raw = (ctypes.c_char * 1024)()
assert M.hipmock_arg(ctypes.c_long(0), 0, raw) == 1024
# the record is the one pointer of the descriptor to nt * nx floats
words = np.frombuffer(raw, dtype=np.uint64)
rec = [int(w) for w in words if w and M.hipmock_size(ctypes.c_void_p(int(w))) == {nt} * {nx} * 4]
assert len(rec) == 1, rec
n = {nt} * {nx}
dev = np.ctypeslib.as_array(ctypes.cast(rec[0], ctypes.POINTER(ctypes.c_float)), (n,))
dev[:] = np.arange(n, dtype=np.int64) % 16777213
d = P.data({nt})
assert np.array_equal(d.ravel(order="F"), dev)
print("ok")
"""


@pytest.mark.parametrize("nt, nx", [(3, 5), (512, 1023), (1024, 512), (2048, 1024), (2049, 1024),
                                    (2048, 2049), (5003, 1021)])
def test_values(nt, nx):
    assert "ok" in hipmock.run(_VALUES.format(nt=nt, nx=nx))


_BUSY = """
import resource, time
V = np.full((8, 3000), 2000.0, order="F")
P = sssi_amd.Propagator(V, 1, 0, 10.0, 10.0, 1e-3)
P.set_points([0], [1], np.zeros(1000))
P.run(1000)
P.data(1000)
M.hipmock_sync_us(300000)
def cpu():
    u = resource.getrusage(resource.RUSAGE_SELF)
    return u.ru_utime + u.ru_stime
a, t = cpu(), time.perf_counter()
P.data(1000)
print((cpu() - a) / (time.perf_counter() - t))
"""


def test_workers_sleep_while_the_gpu_works():
    """A 12 MB result (12 workers) behind 0.3 s of GPU work per wait: the
    call's CPU time stays below a third of one core."""
    assert float(hipmock.run(_BUSY)) < 0.33


_NEW_FAILS = """
V = np.full((8, 3000), 2000.0, order="F")
P = sssi_amd.Propagator(V, 1, 0, 10.0, 10.0, 1e-3)
P.set_points([0], [1], np.zeros(400))
P.run(400)
P.data(400)
out = np.zeros((3000, 400), order="F")
L = sssi_amd.lib()
from sssi_amd._lib import _dp
codes = set()
for k in range(200):
    M.hipmock_fail_new(k)
    rc = L.sssi_prop_get_data(P._h, _dp(out), 400)
    left = M.hipmock_new_left()
    M.hipmock_fail_new(-1)
    codes.add(rc)
    if left >= 0:  # the call made fewer than k allocations
        break
else:
    raise SystemExit("no end")
assert k >= 5 and rc == 0 and codes <= {0, -2}, (k, codes)
# and a handle's creation (velocity scans on threads): 2400 x 3000 cells
V = np.full((2400, 3000), 2000.0, order="F")
h = ctypes.c_void_p()
for k in range(200):
    M.hipmock_fail_new(k)
    rc = L.sssi_prop2d_create(_dp(V), 2400, 3000, 1, 1, 5, 10.0, 10.0, 1e-3, ctypes.byref(h))
    left = M.hipmock_new_left()
    M.hipmock_fail_new(-1)
    assert rc in (0, -2), rc
    if rc == 0: L.sssi_prop_destroy(h)
    if left >= 0: break
assert k >= 5 and rc == 0
print("ok")
"""


def test_failed_host_allocation_is_an_error_code():
    assert "ok" in hipmock.run(_NEW_FAILS)


_POOL = """
import threading
Ps = []
for _ in range(8):
    P = sssi_amd.Propagator(np.full((8, 3000), 2000.0, order="F"), 1, 0, 10.0, 10.0, 1e-3)
    P.set_points([0], [1], np.zeros(1000))
    P.run(1000)
    Ps.append(P)
M.hipmock_sync_us(100000)  # every call holds its chunks while the others start
def once():
    bar = threading.Barrier(8)
    def call(P):
        bar.wait()
        P.data(1000)
    th = [threading.Thread(target=call, args=(P,)) for P in Ps]
    for t in th: t.start()
    for t in th: t.join()
once(); once()
n = M.hipmock_host_mallocs()
for _ in range(3): once()
print(M.hipmock_host_mallocs() - n)
"""


def test_concurrent_calls_find_their_chunks():
    """Eight callers at a time: after the first rounds no pinned memory is
    allocated."""
    assert int(hipmock.run(_POOL)) == 0
