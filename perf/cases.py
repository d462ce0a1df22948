"""Performance cases: what users of sssi_amd run, through its public entry points.

`listed()` names the workloads, `draw()` gives more of the same ranges,
`prepare()` builds what a program holds before the call (models, wavelets,
records, resident handles), `run()` makes one pass, `work()` counts what the
pass cannot do without and `exact()` computes the same outputs in FP64 with
plain torch / numpy.

Host arrays are FP64 because the entry points take MATLAB's arrays: model
upload, run and download are the call for the one-shot entry points, while the
resident handles (Propagator, Rtm2D, Kirchhoff2D, Server) keep their state on
the device between passes.
"""
import math

import numpy as np
import torch

import sssi_amd
from sssi_amd import Kirchhoff2D, Propagator, Rtm2D, Server, helmholtz, synth

# Stability: time steps are this fraction of the staggered scheme's limit.
_CFL = 0.6
_VMIN, _VMAX = 1500.0, 4500.0


def listed():
    return [
        # One shot on the reference's CPU-sized model through the one-shot call,
        # every tenth wavefield kept: launches and host work dominate.
        dict(name="fwd2d_shot_120x240", kind="fwd2d", nz=120, nx=240, N=2, nB=20, nt=1000,
             stride=10),
        # Back-propagation of one record on a small ragged model, with snapshots
        # and the final model: the reverse direction of the same call.
        dict(name="rvs2d_shot_131x275", kind="rvs2d", nz=131, nx=275, N=4, nB=12, nt=600,
             stride=20),
        # The headline forward workload on the resident handle (1000 x 3000 plus
        # damping, nDiffOrder 5): a shot per pass, seismogram to the host.
        dict(name="prop2d_1040x3080", kind="prop2d", nz=1040, nx=3080, N=5, nB=40, nt=1000),
        # The Cerjan-sponge alternative on an ordinary, ragged model.
        dict(name="sponge2d_515x1203", kind="sponge2d", nz=515, nx=1203, N=1, nB=30, nt=800,
             stride=0),
        # A one-shot 3-D forward call on an ordinary grid.
        dict(name="fwd3d_130x140x140", kind="fwd3d", nz=130, nx=140, ny=140, N=4, nB=12, nt=200),
        # The large 3-D forward workload on the resident handle (400^3 plus damping).
        dict(name="prop3d_420x440x440", kind="prop3d", nz=420, nx=440, ny=440, N=4, nB=20, nt=50),
        # Migration of a batch of shots with uneven apertures, BF16 checkpoints,
        # imaging every fifth step, observed data cached as the applications do.
        dict(name="rtm_8shots_600x2400", kind="rtm", nz=600, nx=2400, N=4, nB=30, nt=500, shots=8,
             wmin=400, wmax=1200, img_stride=5, ck="bf16"),
        # A burst of mixed jobs through the serving loop.
        dict(name="serve_burst_6jobs", kind="serve", nz=420, nx=610, n3=128, N=3, nB=20, nt=400),
        # One traveltime table through the eikonal drop-in.
        dict(name="eikonal_101x151", kind="eikonal", nz=101, nx=151, nsrc=1, iMax=126),
        # Traveltime tables of a line of surface positions.
        dict(name="eikonal_300x600_64tables", kind="eikonal", nz=300, nx=600, nsrc=64, iMax=450),
        # Kirchhoff migration of resident records against resident tables.
        dict(name="kirchhoff_300x600_8shots", kind="kirchhoff", nz=300, nx=600, nsr=600, shots=8,
             iMax=100),
        # One frequency of the frequency-domain inversion: 100 sources.
        dict(name="helmholtz_120x140_100src", kind="helmholtz", nz=120, nx=140, N=2, nB=20,
             nsrc=100),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["fwd2d", "rvs2d", "prop2d", "sponge2d", "fwd3d", "prop3d", "rtm",
                       "eikonal", "kirchhoff", "helmholtz"])
    if kind in ("fwd2d", "rvs2d"):
        nz, nx = _log_int(rng, 60, 600), _log_int(rng, 100, 1200)
        return dict(kind=kind, nz=nz, nx=nx, N=rng.randint(1, 8),
                    nB=rng.randint(0, min(40, nz // 3, nx // 3)), nt=_log_int(rng, 150, 1000),
                    stride=rng.choice([0, 10, 25]))
    if kind == "prop2d":
        nz, nx = _log_int(rng, 120, 1040), _log_int(rng, 240, 3080)
        return dict(kind=kind, nz=nz, nx=nx, N=rng.randint(2, 5), nB=rng.randint(10, 40),
                    nt=_log_int(rng, 200, 1000))
    if kind == "sponge2d":
        nz, nx = _log_int(rng, 100, 1040), _log_int(rng, 150, 3080)
        return dict(kind=kind, nz=nz, nx=nx, N=1, nB=rng.randint(0, 40),
                    nt=_log_int(rng, 200, 800), stride=rng.choice([0, 100]))
    if kind in ("fwd3d", "prop3d"):
        n = [_log_int(rng, 48, 200 if kind == "fwd3d" else 320) for _ in range(3)]
        return dict(kind=kind, nz=n[0], nx=n[1], ny=n[2], N=rng.randint(2, 5),
                    nB=rng.randint(0, 16), nt=_log_int(rng, 50, 200) if kind == "fwd3d" else 50)
    if kind == "rtm":
        return dict(kind=kind, nz=_log_int(rng, 150, 600), nx=rng.randint(1200, 2400),
                    N=rng.randint(2, 5), nB=rng.randint(15, 30), nt=_log_int(rng, 200, 500),
                    shots=rng.randint(1, 8), wmin=200, wmax=1200, img_stride=rng.choice([1, 5]),
                    ck=rng.choice(["fp32", "fp16", "bf16"]))
    if kind == "eikonal":
        nz, nx = _log_int(rng, 60, 300), _log_int(rng, 80, 600)
        return dict(kind=kind, nz=nz, nx=nx, nsrc=_log_int(rng, 1, 64), iMax=(nz + nx) // 2)
    if kind == "kirchhoff":
        nx = _log_int(rng, 100, 600)
        return dict(kind=kind, nz=_log_int(rng, 60, 300), nx=nx, nsr=max(2, nx // rng.randint(1, 4)),
                    shots=rng.randint(1, 8), iMax=100)
    nz, nx, N = _log_int(rng, 40, 120), _log_int(rng, 40, 140), rng.randint(1, 3)
    while (2 * N - 1) * nz > 360:  # bands no wider than the listed one's
        N -= 1
    return dict(kind=kind, nz=nz, nx=nx, N=N, nB=min(20, nz // 3, nx // 3),
                nsrc=_log_int(rng, 1, 100))


# --------------------------------------------------------------------- inputs
def _csum(N):
    return float(np.sum(np.abs(synth.dCoef(N))))


def _dt(case, ndim, d):
    s = 1.0 if case["kind"] == "sponge2d" else _csum(case["N"])
    return _CFL * d / (_VMAX * math.sqrt(ndim) * s)


def _model2d(nz, nx, rng):
    """Layers over a lateral trend, 1500-4500 m/s."""
    v = synth.layered_2d(nz, nx, min(8, nz), _VMIN, 4000.0, seed=int(rng.integers(1 << 30)))
    trend = np.cos(np.linspace(0, 2 * np.pi * rng.uniform(0.5, 2), nx) + rng.uniform(0, 6))
    return np.asfortranarray(np.clip(v * (1.0 + 0.06 * trend)[None, :], _VMIN, _VMAX))


def _model3d(nz, nx, ny, rng):
    v = _model2d(nz, nx, rng)
    dip = (np.arange(ny) * rng.uniform(0.02, 0.2)).astype(np.int64)
    out = np.empty((nz, nx, ny), order="F")
    for k in range(ny):
        out[:, :, k] = v[np.minimum(np.arange(nz) + dip[k], nz - 1)]
    return out


def _wavelet(nt, dt, rng):
    f = rng.uniform(0.03, 0.06) / dt  # 17-33 samples per period
    return synth.ricker(f, nt, dt) * rng.uniform(0.5, 2.0)


def _inputs(case, seed):
    """Host inputs of a case, from the seed alone."""
    rng = np.random.default_rng([seed, 77])
    k, d = case["kind"], 10.0
    if k in ("fwd2d", "sponge2d", "prop2d"):
        dt = _dt(case, 2, d)
        nz, nx = case["nz"], case["nx"]
        return dict(v=_model2d(nz, nx, rng), d=d, dt=dt, w=_wavelet(case["nt"], dt, rng),
                    iz=[0], ix=[int(rng.integers(nx // 4, 3 * nx // 4))])
    if k == "rvs2d":
        dt = _dt(case, 2, d)
        nz, nx, nt = case["nz"], case["nx"], case["nt"]
        # a record of a few moveout-like events with noise
        t, x = np.arange(nt)[None, :], np.arange(nx)[:, None]
        data = 0.01 * rng.standard_normal((nx, nt))
        for _ in range(4):
            t0, x0, s = rng.uniform(0.2, 0.8) * nt, rng.uniform(0, nx), rng.uniform(0.4, 1.2)
            tau = (t - np.sqrt(t0 ** 2 + (s * (x - x0)) ** 2)) * (np.pi * 0.045)
            data += (1 - 2 * tau ** 2) * np.exp(-tau ** 2)
        return dict(v=_model2d(nz, nx, rng), d=d, dt=dt, data=np.asfortranarray(data))
    if k in ("fwd3d", "prop3d"):
        dt = _dt(case, 3, d)
        nx, ny = case["nx"], case["ny"]
        return dict(v=_model3d(case["nz"], nx, ny, rng), d=d, dt=dt,
                    w=_wavelet(case["nt"], dt, rng), iz=[0],
                    ix=[int(rng.integers(nx // 4, 3 * nx // 4))],
                    iy=[int(rng.integers(ny // 4, 3 * ny // 4))])
    if k == "rtm":
        dt = _dt(case, 2, d)
        V = _model2d(case["nz"], case["nx"], rng)
        shots = []
        for _ in range(case["shots"]):
            n = int(rng.integers(case["wmin"], case["wmax"] + 1))
            shots.append((int(rng.integers(0, case["nx"] - n + 1)), n, n // 2))
        return dict(V=V, VS=synth.smooth_copy(V, 10), d=d, dt=dt,
                    w=_wavelet(case["nt"], dt, rng), shots=shots)
    if k == "serve":
        jobs = []
        nt, nB = case["nt"], case["nB"]
        for q in range(6):
            sub = np.random.default_rng([seed, 78, q])
            N = case["N"] + q % 2
            if q in (2, 5):
                n = case["n3"] - 9 * (q == 5)
                dt = _CFL * d / (_VMAX * math.sqrt(3) * _csum(N))
                jobs.append(dict(job="fwd3d", v=_model3d(n, n, n, sub), N=N, nB=nB // 2, d=d, dt=dt,
                                 nt=nt // 4, w=_wavelet(nt // 4, dt, sub), src=(0, n // 2, n // 3)))
                continue
            nz, nx = case["nz"] + 37 * q, case["nx"] - 53 * q
            dt = _CFL * d / (_VMAX * math.sqrt(2) * _csum(N))
            v = _model2d(nz, nx, sub)
            if q == 3:
                jobs.append(dict(job="rtm2d", v=v, vs=synth.smooth_copy(v, 5), N=N, nB=nB, d=d,
                                 dt=dt, nt=nt, w=_wavelet(nt, dt, sub), ix=nx // 2))
            else:
                jobs.append(dict(job="fwd2d", v=v, N=N, nB=nB, d=d, dt=dt, nt=nt,
                                 w=_wavelet(nt, dt, sub), ix=nx // 2))
        return dict(jobs=jobs)
    if k == "eikonal":
        nz, nx, n = case["nz"], case["nx"], case["nsrc"]
        V = synth.smooth_copy(_model2d(nz, nx, rng), 4)
        return dict(V=V, d=d, sz=np.ones(n, dtype=np.int64),
                    sx=np.sort(rng.choice(np.arange(1, nx + 1), n, replace=n > nx)))
    if k == "kirchhoff":
        nz, nx, nsr = case["nz"], case["nx"], case["nsr"]
        V = synth.smooth_copy(np.sort(_model2d(nz, nx, rng), axis=0), 10)
        dt = 0.75 * d / float(V.max()) / math.sqrt(2)
        nt = int(round(math.hypot(d * nx, d * nz) * 2.9 / float(V.min()) / dt + 50))
        xsr = np.unique(np.round(np.linspace(1, nx, nsr)).astype(np.int64))
        ixs = np.sort(rng.choice(np.arange(1, xsr.size + 1), case["shots"], replace=False))
        rec = rng.standard_normal((case["shots"], nx, nt), dtype=np.float32)
        # the handle's tables need enough passes for a front to cross the model
        return dict(V=V, d=d, dt=dt, nt=nt, xsr=xsr, ixs=ixs,
                    iMax=max(case["iMax"], (nz + nx) // 4 + 8), rec=rec.astype(np.float64).T)
    if k == "helmholtz":
        nz, nx, nB, n = case["nz"], case["nx"], case["nB"], case["nsrc"]
        m = 1.0 / _model2d(nz, nx, rng) ** 2
        S = np.zeros((nz * nx, n), dtype=np.complex128)
        cols = np.round(np.linspace(nB, nx - 1 - nB, n)).astype(np.int64)
        S[cols * nz, np.arange(n)] = 1.0
        return dict(m=m, S=S, w=2 * np.pi * rng.uniform(6.0, 14.0), d=d)
    raise ValueError(k)


# ------------------------------------------------------------- prepare and run
def prepare(case, seed):
    a = _inputs(case, seed)
    k = case["kind"]
    s = dict(case=case, a=a)
    if k in ("prop2d", "prop3d"):
        extra = dict(dy=a["d"]) if k == "prop3d" else {}
        p = Propagator(a["v"], case["N"], case["nB"], a["d"], a["d"], a["dt"], **extra)
        p.set_points(a["iz"], a["ix"], a["w"], src_iy=a.get("iy"))
        s["prop"] = p
    elif k == "rtm":
        r = Rtm2D(a["V"], a["VS"], case["N"], case["nB"], a["d"], a["d"], a["dt"], case["nt"],
                  img_stride=case["img_stride"], ck_format=case["ck"])
        for xb, xc, ix in a["shots"]:
            r.add_shot(xb, xc, ix, a["w"])
        r.precompute_data()
        s["rtm"] = r
    elif k == "serve":
        s["server"] = Server()
    elif k == "kirchhoff":
        h = Kirchhoff2D(a["V"], a["d"], a["xsr"], a["iMax"], a["dt"])
        h.load_shots(a["rec"])
        a["rec"] = None  # on the device
        s["kirch"] = h
    return s


def run(s):
    case, a = s["case"], s["a"]
    k = case["kind"]
    if k in ("fwd2d", "sponge2d"):
        snap = dict(want_snapshot=case["stride"] > 0, snap_stride=max(1, case["stride"]))
        if k == "fwd2d":
            data, snaps = sssi_amd.fwd_cpml_2d_points(a["v"], case["nt"], case["N"], case["nB"],
                                                      a["d"], a["d"], a["dt"], a["iz"], a["ix"],
                                                      a["w"], **snap)
        else:
            data, snaps = sssi_amd.fwd_sponge_2d_points(a["v"], case["nt"], case["nB"], a["d"],
                                                        a["d"], a["dt"], a["iz"], a["ix"], a["w"],
                                                        **snap)
        return {"data": data} if snaps is None else {"data": data, "snapshots": snaps}
    if k == "rvs2d":
        model, snaps = sssi_amd.rvs_cpml_2d_ex(a["v"], a["data"], case["N"], case["nB"], a["d"],
                                               a["d"], a["dt"], want_snapshot=case["stride"] > 0,
                                               snap_stride=max(1, case["stride"]))
        return {"model": model} if snaps is None else {"model": model, "snapshots": snaps}
    if k == "fwd3d":
        data, _ = sssi_amd.fwd_cpml_3d_points(a["v"], case["nt"], case["N"], case["nB"], a["d"],
                                              a["d"], a["d"], a["dt"], a["iz"], a["ix"], a["iy"],
                                              a["w"])
        return {"data": data}
    if k in ("prop2d", "prop3d"):
        p = s["prop"]
        p.reset()
        p.run(case["nt"])
        return {"data": p.data(case["nt"])}
    if k == "rtm":
        s["rtm"].migrate(batched=True)
        return {"stack": s["rtm"].stack()}
    if k == "serve":
        srv, ids = s["server"], []
        for j in a["jobs"]:
            if j["job"] == "fwd3d":
                ids.append(srv.submit_fwd3d(j["v"], j["nt"], j["N"], j["nB"], j["d"], j["d"],
                                            j["d"], j["dt"], j["src"], j["w"]))
            elif j["job"] == "rtm2d":
                ids.append(srv.submit_rtm2d(j["v"], j["vs"], j["nt"], j["N"], j["nB"], j["d"],
                                            j["d"], j["dt"], j["ix"], j["w"], img_stride=5,
                                            ck_format="bf16"))
            else:
                ids.append(srv.submit_fwd2d(j["v"], j["nt"], j["N"], j["nB"], j["d"], j["d"],
                                            j["dt"], 0, j["ix"], j["w"]))
        for i in ids:
            srv.wait(i)
        return [srv.result(i) for i in ids]
    if k == "eikonal":
        if case["nsrc"] == 1:
            return {"T": sssi_amd.eikonal2d(a["V"], a["d"], int(a["sz"][0]), int(a["sx"][0]),
                                            case["iMax"])}
        return {"T": sssi_amd.eikonal2d_batch(a["V"], a["d"], a["sz"], a["sx"], case["iMax"])}
    if k == "kirchhoff":
        return {"stack": s["kirch"].migrate_loaded(a["xsr"], a["ixs"])}
    return {"U": helmholtz.solve(a["m"], a["S"], a["w"], case["N"], case["nB"], a["d"], a["d"])}


# ------------------------------------------------------------------------ work
# Field levels and model that fit the chip's LDS need not go to memory between
# time steps; larger ones are streamed once per step (two levels and v^2 dt^2
# read, one level written, FP32).
_ON_CHIP = 32e6


def _steps(cells, ndim, L, nt, results):
    stream = 16.0 * cells * nt if 12.0 * cells > _ON_CHIP else 16.0 * cells
    return {"bytes": stream + results, "flops": float(nt) * cells * (3 * ndim * L + 6)}


def work(case):
    k = case["kind"]
    if k in ("fwd2d", "rvs2d", "prop2d", "sponge2d"):
        cells, nt = case["nz"] * case["nx"], case["nt"]
        snaps = -(-nt // case["stride"]) if case.get("stride", 0) > 0 else 0
        return _steps(cells, 2, 2 * case["N"] - 1, nt, 8.0 * (nt * case["nx"] + snaps * cells))
    if k in ("fwd3d", "prop3d"):
        return _steps(case["nz"] * case["nx"] * case["ny"], 3, 2 * case["N"] - 1, case["nt"],
                      8.0 * case["nt"] * case["nx"] * case["ny"])
    if k == "rtm":
        width = (case["wmin"] + case["wmax"]) / 2 + 2 * case["nB"]
        cells = case["shots"] * (case["nz"] + case["nB"]) * width
        L, nck = 2 * case["N"] - 1, -(-case["nt"] // case["img_stride"])
        # forward and reverse propagation; checkpoints written and read, the
        # two image sums updated at each
        w = _steps(cells, 2, L, 2 * case["nt"], 8.0 * case["nz"] * case["nx"])
        ck = 4 if case["ck"] == "fp32" else 2
        return {"bytes": w["bytes"] + cells * nck * (2.0 * ck + 16.0), "flops": w["flops"]}
    if k == "serve":
        total = {"bytes": 0.0, "flops": 0.0}
        for q in range(6):
            N = case["N"] + q % 2
            if q in (2, 5):
                n = case["n3"] - 9 * (q == 5)
                w = _steps(float(n) ** 3, 3, 2 * N - 1, case["nt"] // 4, 8.0 * n * n * (case["nt"] // 4))
            else:
                cells = (case["nz"] + 37 * q) * (case["nx"] - 53 * q)
                w = _steps(cells, 2, 2 * N - 1, case["nt"] * (3 if q == 3 else 1), 8.0 * cells)
            total = {x: total[x] + w[x] for x in total}
        return total
    if k == "eikonal":
        cells = float(case["nz"] * case["nx"] * case["nsrc"])
        stream = 4 * case["iMax"] if 16.0 * cells > _ON_CHIP else 1
        return {"bytes": 8.0 * case["nz"] * case["nx"] + 16.0 * cells * stream,
                "flops": cells * 4 * case["iMax"] * 14.0}
    if k == "kirchhoff":
        cells = float(case["nz"] * case["nx"])
        sums = cells * case["nsr"] * case["shots"]
        # index tables and records read once, image written
        nt = math.hypot(case["nx"], case["nz"]) * 12
        return {"bytes": 4.0 * cells * (case["nsr"] + case["shots"]) +
                8.0 * case["shots"] * case["nx"] * nt + 8.0 * cells, "flops": 2.0 * sums}
    n = float(case["nz"] * case["nx"])
    kl = (2 * case["N"] - 1) * case["nz"]
    # banded LU (complex, pivoting widens U to 2 kl) and two sweeps per source;
    # the factors are written and read once
    return {"bytes": 2 * 16.0 * n * 3 * kl + 32.0 * n * case["nsrc"],
            "flops": 8.0 * n * (kl * 2.0 * kl + 3.0 * kl * case["nsrc"])}


# ------------------------------------------------------------- FP64 references
_DEV = "cuda" if torch.cuda.is_available() else "cpu"


def _t(x):
    return torch.as_tensor(np.ascontiguousarray(x), dtype=torch.float64, device=_DEV)


def _damp(u, v, length):
    return -(3.0 * v) / (2.0 * length) * math.log(1e-6) * (u / length) ** 2


class _Cpml:
    """CPML propagation, full-grid memory variables, index order [z, x(, y)]."""

    def __init__(self, v, N, nB, d, dt):
        v = _t(v)
        self.n, self.N, self.dim = v.shape, N, v.dim()
        self.c = [float(c) / d for c in synth.dCoef(N)]
        self.v2 = (v * dt) ** 2
        self.b = []
        for ax in range(self.dim):
            prof = torch.zeros_like(v)
            if nB:
                n = v.shape[ax]
                if self.dim == 2:
                    src, unit = v, d
                else:  # 3-D: index units; x and z profiles from the first y slice, y from the top
                    src = v[:, :, :1].expand_as(v) if ax < 2 else v[:1].expand_as(v)
                    unit = 1.0
                up = [1] * self.dim
                up[ax] = nB
                rise = (torch.arange(1, nB + 1, device=_DEV, dtype=torch.float64) * unit).view(up)
                hi = [slice(None)] * self.dim
                hi[ax] = slice(n - nB, n)
                prof[tuple(hi)] = _damp(rise, src[tuple(hi)], nB * unit)
                if ax > 0:  # no damping at the free surface
                    lo = [slice(None)] * self.dim
                    lo[ax] = slice(0, nB)
                    prof[tuple(lo)] = _damp(rise.flip(ax), src[tuple(lo)], nB * unit)
            self.b.append(torch.exp(-prof * dt))
        z = torch.zeros_like(v)
        self.phi = [z.clone() for _ in range(self.dim)]
        self.psi = [z.clone() for _ in range(self.dim)]
        self.p, self.po = z, z.clone()

    def step(self, add):
        N, L = self.N, 2 * self.N - 1
        P = torch.zeros_like(self.p)
        for ax in range(self.dim):
            n = self.n[ax]
            pad = [0, 0] * self.dim
            pad[2 * (self.dim - 1 - ax)] = pad[2 * (self.dim - 1 - ax) + 1] = L
            q = torch.nn.functional.pad(self.p, pad)
            m = n + 2 * N - 1  # half points -N .. n+N-2
            A = torch.zeros_like(q.narrow(ax, 0, m))
            for k, c in enumerate(self.c):
                A.add_(q.narrow(ax, N + k, m), alpha=c)
                A.sub_(q.narrow(ax, N - 1 - k, m), alpha=c)
            b = self.b[ax]
            self.phi[ax].mul_(b).addcmul_(b - 1, A.narrow(ax, N, n))
            A.narrow(ax, N, n).add_(self.phi[ax])
            D = torch.zeros_like(self.p)
            for k, c in enumerate(self.c):
                D.add_(A.narrow(ax, N + k, n), alpha=c)
                D.sub_(A.narrow(ax, N - 1 - k, n), alpha=c)
            self.psi[ax].mul_(b).addcmul_(b - 1, D)
            P.add_(D).add_(self.psi[ax])
        add(P)
        self.po = P.mul_(self.v2).add_(self.p, alpha=2.0).sub_(self.po)
        self.p, self.po = self.po, self.p


def _forward(g, nt, cell, w, each=None):
    """Point-source forward run; receivers on the top row / plane."""
    data = []
    for t in range(nt):
        def add(P, a=float(w[t])):
            P[cell] += a
        g.step(add)
        data.append(g.p[0].clone())
        if each:
            each(t, g.p)
    return torch.stack(data, dim=-1)


def _reverse(g, data, each=None):
    for t in range(data.shape[1] - 1, -1, -1):
        def add(P, row=data[:, t]):
            P[0] += row
        g.step(add)
        if each:
            each(t, g.p)


def _kept(stride):
    kept = []
    return kept, (lambda t, p: kept.append(p.clone()) if t % stride == 0 else None)


def _np(x):
    return x.cpu().numpy()


def _rtm_image(V, VS, N, nB, d, dt, nt, w, ix, stride, eps=1e-3):
    fs, keep = _kept(stride)
    cell = (0, ix)
    dtrue = _forward(_Cpml(V, N, nB, d, dt), nt, cell, w)
    dsmooth = _forward(_Cpml(VS, N, nB, d, dt), nt, cell, w, keep)
    num, den = torch.zeros_like(fs[0]), torch.zeros_like(fs[0])

    def image(t, p):
        if t % stride == 0:
            f = fs[t // stride]
            num.addcmul_(f, p)
            den.addcmul_(f, f)
    _reverse(_Cpml(V, N, nB, d, dt), dtrue - dsmooth, image)
    return num / (eps + den)


def _sponge(case, a):
    v, d, dt, nB = _t(a["v"]), a["d"], a["dt"], case["nB"]
    nz, nx = v.shape
    g = torch.ones_like(v)
    f = torch.tensor([math.exp(-((0.015 * (nB - m)) ** 2)) ** 10 for m in range(nB)],
                     device=_DEV, dtype=torch.float64)
    if nB:
        g[:, :nB] = f[None, :]
        g[:, nx - nB:] = f.flip(0)[None, :]
        g[nz - nB:, :] = f.flip(0)[:, None]
    a2 = (v * dt / d) ** 2
    p1, p2 = torch.zeros_like(v), torch.zeros_like(v)
    data, snaps = [], []
    for t in range(case["nt"]):
        q = torch.nn.functional.pad(p2, (1, 1, 1, 1))
        lap = q[1:-1, 2:] + q[1:-1, :-2] + q[2:, 1:-1] + q[:-2, 1:-1] - 4.0 * p2
        p3 = 2.0 * p2 - p1 + a2 * lap
        p3[a["iz"][0], a["ix"][0]] -= (a2[a["iz"][0], a["ix"][0]] * d * d) * float(a["w"][t])
        p1, p2 = p2 * g, p3 * g
        data.append(p2[0].clone())
        if case["stride"] and t % case["stride"] == 0:
            snaps.append(p2.clone())
    out = {"data": _np(torch.stack(data, dim=-1))}
    if snaps:
        out["snapshots"] = _np(torch.stack(snaps, dim=-1))
    return out


def _eikonal(V, d, sz, sx, iMax):
    """Tables [source, z, x]: the reference's Jacobi passes."""
    s = 1.0 / _t(V)
    nz, nx = s.shape
    n = len(sz)
    k = torch.arange(n, device=_DEV)
    iz = torch.as_tensor(np.asarray(sz) - 1, device=_DEV)
    ix = torch.as_tensor(np.asarray(sx) - 1, device=_DEV)
    T = torch.full((n, nz, nx), 65535.0, dtype=torch.float64, device=_DEV)
    T[k, iz, ix] = 0.0
    sd = s * float(int(d))
    sd2 = 2.0 * sd * sd
    for _ in range(4 * iMax):
        q = torch.cat([T[:, 1:2], T, T[:, -2:-1]], dim=1)
        a = torch.minimum(q[:, :-2], q[:, 2:])
        q = torch.cat([T[:, :, 1:2], T, T[:, :, -2:-1]], dim=2)
        b = torch.minimum(q[:, :, :-2], q[:, :, 2:])
        e = a - b
        two = 0.5 * (a + b + torch.sqrt(torch.clamp(sd2 - e * e, min=0.0)))
        N = torch.minimum(T, torch.where(e.abs() < sd, two, torch.minimum(a, b) + sd))
        N[k, iz, ix] = 0.0
        if torch.equal(N, T):
            break  # further passes change nothing
        T = N
    return T


def _kirchhoff(case, seed):
    a = _inputs(case, seed)
    T = _eikonal(a["V"], a["d"], np.ones(a["xsr"].size, dtype=np.int64), a["xsr"], a["iMax"])
    r = T / a["dt"]
    idx = torch.floor(r + 0.5).to(torch.int64) + 1  # round half away from zero (T >= 0)
    stack = torch.zeros_like(T[0])
    for q, i in enumerate(a["ixs"]):
        rec = _t(a["rec"][:, :, q])
        acc = torch.zeros_like(stack)
        for r in range(a["xsr"].size):
            acc += rec[:, int(a["xsr"][r]) - 1][idx[int(i) - 1] + idx[r] - 1]
        stack += acc
    return {"stack": _np(stack)}


def _helmholtz(case, a):
    """Impedance matrix in blocks of k = 2N-1 columns of cells, block
    tridiagonal elimination, one step of refinement."""
    m, S, w, d = a["m"], a["S"], a["w"], a["d"]
    nz, nx = m.shape
    N, nB = case["N"], case["nB"]
    k, v = 2 * N - 1, np.sqrt(1.0 / m)
    xd, zd = np.zeros((nz, nx)), np.zeros((nz, nx))
    if nB:
        u = np.arange(1, nB + 1) * d
        xd[:, nx - nB:] = _damp(u[None, :], v[:, nx - nB:], nB * d)
        xd[:, :nB] = _damp(u[::-1][None, :], v[:, :nB], nB * d)
        zd[nz - nB:] = _damp(u[:, None], v[nz - nB:], nB * d)
    c, f = synth.dCoef(N), np.zeros(2 * k + 1)
    for i in range(1, N + 1):
        for j in range(1, N + 1):
            p = c[i - 1] * c[j - 1]
            f[k + i + j - 1] += p
            f[k - (i + j - 1)] += p
            f[k + i - j] -= p
            f[k - (i - j)] -= p
    fz, fx = ((1j * w / (d * (1j * w + q))) ** 2 for q in (zd, xd))
    nb, bs = -(-nx // k), k * nz
    lo, di, up = [], [], []
    for b in range(nb):
        cols = list(range(b * k, min(nx, b * k + k)))
        n = len(cols) * nz
        D = np.zeros((n, n), dtype=np.complex128)
        Lm = np.zeros((n, bs), dtype=np.complex128)
        U = np.zeros((n, max(0, min(nx, b * k + 2 * k) - (b * k + k)) * nz), dtype=np.complex128)
        for q, j in enumerate(cols):
            i = np.arange(nz)
            r = q * nz + i
            D[r, r] += m[:, j] * w * w + f[k] * (fz[:, j] + fx[:, j])
            for o in range(1, k + 1):
                D[r[o:], r[o:] - o] += f[k - o] * fz[o:, j]
                D[r[:nz - o], r[:nz - o] + o] += f[k + o] * fz[:nz - o, j]
                for jj, e in ((j - o, f[k - o]), (j + o, f[k + o])):
                    if not 0 <= jj < nx:
                        continue
                    bb, rr = divmod(jj, k)
                    M = D if bb == b else Lm if bb < b else U
                    M[r, rr * nz + i] += e * fx[:, j]
        lo.append(Lm)
        di.append(D)
        up.append(U)

    def parts(X):
        return [X[b * bs:(b + 1) * bs] for b in range(nb)]

    def times(X):
        x = parts(X)
        return np.concatenate([di[b] @ x[b] + (lo[b] @ x[b - 1] if b else 0) +
                               (up[b] @ x[b + 1] if b + 1 < nb else 0) for b in range(nb)])
    inv = []
    for b in range(nb):
        D = di[b] - lo[b] @ inv[-1] @ up[b - 1] if b else di[b]
        inv.append(np.linalg.inv(D))

    def solve(R):
        y, r = [], parts(R)
        for b in range(nb):
            y.append(r[b] - lo[b] @ (inv[b - 1] @ y[-1]) if b else r[b])
        x = [None] * nb
        for b in range(nb - 1, -1, -1):
            x[b] = inv[b] @ (y[b] - (up[b] @ x[b + 1] if b + 1 < nb else 0))
        return np.concatenate(x)
    X = solve(-S)
    X = X + solve(-S - times(X))
    return {"U": np.asfortranarray(X + solve(-S - times(X)))}


def exact(case, seed):
    k = case["kind"]
    if k == "kirchhoff":
        return _kirchhoff(case, seed)
    a = _inputs(case, seed)
    if k in ("fwd2d", "prop2d", "fwd3d", "prop3d"):
        g = _Cpml(a["v"], case["N"], case["nB"], a["d"], a["dt"])
        cell = (a["iz"][0], a["ix"][0]) + ((a["iy"][0],) if "iy" in a else ())
        kept, keep = _kept(max(1, case.get("stride", 0)))
        data = _forward(g, case["nt"], cell, a["w"], keep if case.get("stride", 0) else None)
        out = {"data": _np(data)}
        if kept:
            out["snapshots"] = _np(torch.stack(kept, dim=-1))
        return out
    if k == "rvs2d":
        g, L = _Cpml(a["v"], case["N"], case["nB"], a["d"], a["dt"]), 2 * case["N"] - 1
        kept, keep = _kept(max(1, case["stride"]))
        _reverse(g, _t(a["data"]), keep if case["stride"] else None)
        out = {"model": np.pad(_np(g.po), L)}  # the field one step before the last
        if kept:
            out["snapshots"] = _np(torch.stack(kept[::-1], dim=-1))
        return out
    if k == "sponge2d":
        return _sponge(case, a)
    if k == "rtm":
        stack, nB = np.zeros((case["nz"], case["nx"])), case["nB"]
        for xb, xc, ix in a["shots"]:
            V, VS = (synth.extBoundary(M[:, xb:xb + xc], nB, 2) for M in (a["V"], a["VS"]))
            img = _np(_rtm_image(V, VS, case["N"], nB, a["d"], a["dt"], case["nt"], a["w"],
                                 ix + nB, case["img_stride"]))
            stack[:, xb:xb + xc] += img[:case["nz"], nB:nB + xc]
        return {"stack": stack}
    if k == "serve":
        out = []
        for j in a["jobs"]:
            if j["job"] == "rtm2d":
                out.append(_np(_rtm_image(j["v"], j["vs"], j["N"], j["nB"], j["d"], j["dt"],
                                          j["nt"], j["w"], j["ix"], 5)))
                continue
            g = _Cpml(j["v"], j["N"], j["nB"], j["d"], j["dt"])
            cell = j["src"] if j["job"] == "fwd3d" else (0, j["ix"])
            out.append(_np(_forward(g, j["nt"], cell, j["w"])))
        return out
    if k == "eikonal":
        T = _eikonal(a["V"], a["d"], a["sz"], a["sx"], case["iMax"])
        return {"T": _np(T[0] if case["nsrc"] == 1 else T.permute(1, 2, 0))}
    return _helmholtz(case, a)
