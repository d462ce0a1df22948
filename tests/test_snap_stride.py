"""Snapshot strides beyond the last step keep the first wavefield alone, also
those that do not fit 32 bits: what the launches are told, without a GPU, and
the same snapshots as at a stride of nt on one."""
import numpy as np
import pytest

import hipmock
import sssi_amd
from sssi_amd import synth

STRIDES = [25, 2 ** 31, 2 ** 32, 2 ** 32 + 1, 2 ** 63 - 1]

_SPONGE = """
class A(ctypes.Structure):  # Sponge2dArgs
    _fields_ = [("p", ctypes.c_void_p * 6), ("grid", ctypes.c_int * 5), ("f", ctypes.c_float * 2),
                ("t", ctypes.c_int * 3), ("src", ctypes.c_void_p * 2), ("ns", ctypes.c_int * 2),
                ("surf", ctypes.c_void_p), ("surf_nt", ctypes.c_int), ("rec", ctypes.c_void_p),
                ("snap", ctypes.c_void_p), ("stride", ctypes.c_int), ("slot0", ctypes.c_int64)]
watch("sponge2d_steps", ctypes.sizeof(A))
v = np.full((30, 40), 2000.0, order="F")
d, s = sssi_amd.fwd_sponge_2d_points(v, 25, 5, 10.0, 10.0, 1e-3, [0], [20],
                                     synth.ricker(20.0, 25, 1e-3), want_snapshot=True,
                                     snap_stride={stride})
assert s.shape == (30, 40, 1)
for k in range(count("sponge2d_steps")):
    a = arg(k, 0, A)
    hit = [t for t in range(a.t[0], a.t[0] + a.t[2]) if a.stride != 0 and t % a.stride == 0]
    assert a.snap and a.stride != 0 and a.slot0 == 0 and hit in ([], [0]), (a.stride, hit)
print("ok")
"""


@pytest.mark.parametrize("stride", STRIDES)
def test_what_the_sponge_is_told(stride):
    assert "ok" in hipmock.run(_SPONGE.format(stride=stride), timeout=30)


@pytest.mark.gpu
@pytest.mark.parametrize("stride", STRIDES[1:])
@pytest.mark.parametrize("kind", ["fwd", "rvs", "sponge", "rvs_sponge", "3d"])
def test_first_wavefield_alone(kind, stride):
    nt, dt = 25, 1e-3
    w = synth.ricker(40.0, nt, dt)
    rng = np.random.default_rng(5)
    v = np.asfortranarray(1500.0 + 1000.0 * rng.random((40, 70)))
    rec = np.asfortranarray(rng.standard_normal((70, nt)))
    v3 = np.asfortranarray(1500.0 + 1000.0 * rng.random((20, 30, 24)))

    def run(st):
        k = dict(want_snapshot=True, snap_stride=st)
        if kind == "fwd":
            return sssi_amd.fwd_cpml_2d_points(v, nt, 2, 5, 10.0, 10.0, dt, [0], [30], w, **k)
        if kind == "rvs":
            return sssi_amd.rvs_cpml_2d_ex(v, rec, 2, 5, 10.0, 10.0, dt, **k)
        if kind == "sponge":
            return sssi_amd.fwd_sponge_2d_points(v, nt, 5, 10.0, 10.0, dt, [0], [30], w, **k)
        if kind == "rvs_sponge":
            return sssi_amd.rvs_sponge_2d_ex(v, rec, 5, 10.0, 10.0, dt, **k)
        return sssi_amd.fwd_cpml_3d_points(v3, nt, 2, 4, 10.0, 10.0, 10.0, dt, [0], [15], [12], w,
                                           **k)
    print(f"stride {stride} {kind}", flush=True)
    a, s = run(stride)
    b, r = run(nt)
    assert np.array_equal(a, b) and np.array_equal(s, r)
    assert s.shape[-1] == 1 and np.any(a != 0)
