"""Performance cases of the framework: the calls that its users' programs spend their time in.

listed() are fixed cases, draw(rng) gives further ones of the same ranges, prepare() makes what a program holds before the
call, run() is one pass through public entry points, work() is what a pass cannot do without, and exact() is the same
pass in plain 64-bit torch.

Kinds:
  solve     hydro.fluid_solver on device arrays: one Flu_AdvanceDt call.  From a handful of patch groups (a small refined
            level, latency) to the 4096 of the benchmark; both schemes, precisions, the three Riemann solvers, a run-time
            limiter, with and without the coarse-fine fluxes and the fused CFL time step
  batch     hydro.solve_batch: the patch groups of three AMR levels, each with its own dt and dh, as one work-queue launch
  uniform   hydro.UniformLevel.step: ghost zones, solve, copy back, next dt of a periodic level
  twolevel  amr.TwoLevel.step: base step, two refined substeps with interpolated ghost zones, restriction, flux fix-up
  adjoint   hydro.mhm_adjoint: the vector-Jacobian product of a step
  tangent   hydro.mhm_tangent: the Jacobian-vector product of a step
  rollout   diff.rollout forward and backward: the gradient of a loss after several steps
  host      hydro_asyn_fluid_solver on pinned host arrays: the drop-in call of a CPU-resident code, copies included
"""
import ctypes
import math

import torch

from gamer_amd import amr, diff, hydro

DEV = "cuda:0"
GAMMA = 5.0 / 3.0
FLOAT = {"f32": torch.float32, "f64": torch.float64}
PRECISION = {"f32": "fp32", "f64": "fp64"}


# ---------------------------------------------------------------- cases

def _solve(npg, dtype, scheme="MHM_RP", rsolver="HLLC", limiter="VL_GMINMOD", flux=True, dt=False):
    return {"kind": "solve", "npg": npg, "dtype": dtype, "scheme": scheme, "rsolver": rsolver, "limiter": limiter,
            "flux": flux, "dt": dt}


def listed():
    return [
        # a small refined level: 8 patch groups, far fewer than the chip has compute units
        {"name": "solve_f32_8", **_solve(8, "f32")},
        # the benchmark workload: 4096 patch groups, 256^3 cells
        {"name": "solve_f32_4096", **_solve(4096, "f32")},
        # a double-precision level of an odd size, with the CFL time step of the next step computed in the solver
        {"name": "solve_f64_1331", **_solve(1331, "f64", dt=True)},
        # the most expensive solver with a limiter chosen at run time, on a ragged level
        {"name": "solve_f64_roe_300", **_solve(300, "f64", rsolver="ROE", limiter="VANLEER")},
        # the Hancock scheme with the HLLE solver, no coarse-fine boundary
        {"name": "solve_f32_mhm_1000", **_solve(1000, "f32", scheme="MHM", rsolver="HLLE", flux=False)},
        # three AMR levels of one hierarchy in one launch
        {"name": "batch_f32_8704", "kind": "batch", "n0": 512, "n1": 2048, "n2": 6144, "dtype": "f32"},
        # one step of a periodic level without refinement
        {"name": "uniform_f32_192x160x128", "kind": "uniform", "gx": 12, "gy": 10, "gz": 8, "dtype": "f32", "scheme": "MHM_RP"},
        # base level of 128^3 cells whose central half is refined: the AMR step
        {"name": "twolevel_f32_128", "kind": "twolevel", "nx": 16, "ny": 16, "nz": 16, "lx": 4, "ly": 4, "lz": 4,
         "mx": 8, "my": 8, "mz": 8, "dtype": "f32"},
        # reverse mode of one step
        {"name": "adjoint_f64_512", "kind": "adjoint", "npg": 512, "rsolver": "HLLC"},
        # forward mode of one step on a smaller, odd level
        {"name": "tangent_f64_125", "kind": "tangent", "npg": 125, "rsolver": "HLLC"},
        # gradient of a 4-step rollout on 64^3 cells
        {"name": "rollout_f64_64", "kind": "rollout", "gx": 4, "gy": 4, "gz": 4, "steps": 4},
        # the host-array call of a CPU code: pinned arrays in and out over 4 streams
        {"name": "host_f32_512", "kind": "host", "npg": 512, "dtype": "f32", "streams": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve"] * 7 + ["batch", "uniform", "uniform", "twolevel", "adjoint", "tangent", "rollout", "host"])
    dtype = rng.choice(["f32", "f32", "f64"])
    if kind == "solve":
        return _solve(_log_int(rng, 1, 4096 if dtype == "f32" else 2048), dtype, rng.choice(["MHM_RP", "MHM_RP", "MHM"]),
                      rng.choice(["HLLC", "HLLC", "HLLE", "ROE"]), rng.choice(["VL_GMINMOD", "VL_GMINMOD", "VANLEER", "GMINMOD"]),
                      rng.random() < 0.75, rng.random() < 0.4)
    if kind == "batch":
        return {"kind": kind, "n0": _log_int(rng, 8, 512), "n1": _log_int(rng, 16, 1024), "n2": _log_int(rng, 16, 2048),
                "dtype": dtype}
    if kind == "uniform":
        return {"kind": kind, "gx": rng.randint(1, 10), "gy": rng.randint(1, 9), "gz": rng.randint(1, 8), "dtype": dtype,
                "scheme": rng.choice(["MHM_RP", "MHM_RP", "MHM"])}
    if kind == "twolevel":
        n = [2 * rng.randint(2, 7) for _ in range(3)]
        m = [rng.randint(1, k - 2) for k in n]
        at = [rng.randint(1, k - j - 1) for k, j in zip(n, m)]
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "lx": at[0], "ly": at[1], "lz": at[2], "mx": m[0],
                "my": m[1], "mz": m[2], "dtype": dtype}
    if kind in ("adjoint", "tangent"):
        return {"kind": kind, "npg": _log_int(rng, 1, 512), "rsolver": rng.choice(["HLLC", "HLLC", "HLLE", "ROE"])}
    if kind == "rollout":
        return {"kind": kind, "gx": rng.randint(1, 4), "gy": rng.randint(1, 4), "gz": rng.randint(1, 4), "steps": rng.randint(1, 4)}
    return {"kind": kind, "npg": _log_int(rng, 4, 512), "dtype": dtype, "streams": rng.choice([1, 2, 4, 4, 8])}


# ---------------------------------------------------------------- inputs

def _cons(rho, v, p):
    return torch.stack([rho, rho * v[0], rho * v[1], rho * v[2],
                        p / (GAMMA - 1.0) + 0.5 * rho * (v[0] ** 2 + v[1] ** 2 + v[2] ** 2)])


def _signal_speed(cons):
    """max_d(|v_d| + c_s) of every cell, (5, ...) -> (...)."""
    p = (GAMMA - 1.0) * (cons[4] - 0.5 * (cons[1] ** 2 + cons[2] ** 2 + cons[3] ** 2) / cons[0])
    return cons[1:4].abs().amax(0) / cons[0] + torch.sqrt(GAMMA * p / cons[0])


def _cfl_dt(cons, dh, cfl=0.5):
    return cfl * dh / _signal_speed(cons).max().item()


def _medium(shape, seed, sod=True):
    """A periodic (5, Z, Y, X) gas: lognormal density and pressure, velocities of 0.3 sound speeds; with ``sod`` its first
    half along x holds a Sod plane every 16 cells and every 16th block of 16 cells a pressure spike."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    new = lambda: torch.randn(shape, generator=g, dtype=torch.float64, device=DEV)  # noqa: E731
    rho, p = torch.exp(0.5 * new()), torch.exp(0.5 * new())
    cs = torch.sqrt(GAMMA * p / rho)
    v = [0.3 * cs * new() for _ in range(3)]
    if sod:
        x = torch.arange(shape[2], device=DEV)
        half, left = (x < shape[2] // 2).expand(shape), (x % 16 < 8).expand(shape)
        rho = torch.where(half, torch.where(left, 1.0, 0.125).to(rho.dtype), rho)
        p = torch.where(half, torch.where(left, 1.0, 0.1).to(p.dtype), p)
        v = [torch.where(half, 0.0, w) for w in v]
        at = torch.randint(0, 16, (shape[2] // 256 + 1, 3), generator=g, device=DEV)
        k = torch.arange(at.shape[0], device=DEV) * 256
        p[at[:, 0], at[:, 1], (k + at[:, 2]) % shape[2]] *= 1.0e3
    return _cons(rho, v, p)


def _smooth(shape, seed, noise=0.0):
    """A periodic gas of a few sine modes with random phases; ``noise``: lognormal scatter of density and pressure."""
    g = torch.Generator().manual_seed(seed)
    z, y, x = torch.meshgrid(*((torch.arange(n, dtype=torch.float64) + 0.5) / n for n in shape), indexing="ij")
    x, y, z = x.to(DEV), y.to(DEV), z.to(DEV)

    def mode(most):
        k = torch.randint(1, most + 1, (3,), generator=g).tolist()
        ph = 6.283185307179586 * torch.rand((), generator=g).item()
        return torch.sin(6.283185307179586 * (k[0] * x + k[1] * y + k[2] * z) + ph)

    rho = 1.0 + 0.1 * mode(3) + 0.05 * mode(3)
    p = 1.0 + 0.1 * mode(2)
    v = [0.3 * mode(2) for _ in range(3)]
    if noise:
        gd = torch.Generator(device=DEV).manual_seed(seed)
        rho = rho * torch.exp(noise * torch.randn(shape, generator=gd, dtype=torch.float64, device=DEV))
        p = p * torch.exp(noise * torch.randn(shape, generator=gd, dtype=torch.float64, device=DEV))
    return _cons(rho, v, p)


def _cut(cons, ghost):
    """Periodic (5, Z, Y, X) -> patch-group blocks (npg, 5, N, N, N), x fastest."""
    n = 16 + 2 * ghost
    g = cons
    for d in (1, 2, 3):
        m = cons.shape[d]
        g = g.index_select(d, torch.arange(-ghost, m + ghost, device=cons.device) % m)
    b = g.unfold(1, n, 16).unfold(2, n, 16).unfold(3, n, 16)
    return b.permute(1, 2, 3, 0, 4, 5, 6).reshape(-1, 5, n, n, n).contiguous()


def _ghost(scheme):
    return 3 if scheme == "MHM_RP" else 2


def _groups(npg, seed, scheme="MHM_RP", sod=True):
    """npg patch-group inputs in a row, and the dt and dh of their level."""
    cons = _medium((16, 16, 16 * npg), seed, sod)
    dh = 1.0 / 256.0
    return _cut(cons, _ghost(scheme)), _cfl_dt(cons, dh), dh


def _levels(case, seed):
    """Patch groups of three levels, refinement ratio 2 (dh and dt halve), mixed in proportion to the level sizes."""
    n = [case["n0"], case["n1"], case["n2"]]
    u, dts = zip(*((b, t * 2 ** l) for l, (b, t) in enumerate(_groups(k, seed + 7 * l)[:2] for l, k in enumerate(n))))
    dt = 0.5 * min(dts)                  # dh is the same for the three media; level l takes dt / 2^l on dh / 2^l
    dtdh = torch.cat([torch.tensor([[dt / 2 ** l, 1.0 / 256.0 / 2 ** l]], dtype=torch.float64).expand(k, 2) for l, k in enumerate(n)])
    key = torch.cat([(torch.arange(k, dtype=torch.float64) + 0.5) / k for k in n])
    order = torch.argsort(key, stable=True)
    return torch.cat(u)[order.to(DEV)], dtdh[order].contiguous().to(DEV)


def _two_level(case, seed):
    """Base level (5, Z, Y, X) with a refined box of base patches, the refined cells injected from their base cells."""
    shape = [8 * case[k] for k in ("nz", "ny", "nx")]
    base = _smooth(shape, seed, noise=0.1)
    lo = [8 * case[k] for k in ("lz", "ly", "lx")]
    m = [8 * case[k] for k in ("mz", "my", "mx")]
    box = base[:, lo[0]:lo[0] + m[0], lo[1]:lo[1] + m[1], lo[2]:lo[2] + m[2]]
    fine = box.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)
    dh = 1.0 / shape[2]
    return base, fine, 0.5 * _cfl_dt(base, dh), dh, lo, m


_API = {}


def _host_api(npg, dtype, streams):
    """The device buffers and streams of the host-array call: one set at a time, as the library holds them."""
    key = (npg, dtype, streams)
    if _API.get("key") != key:
        if "key" in _API:
            _API["api"].free()
        _API["api"], _API["key"] = hydro.GpuFluidApi(npg, gpu_nstream=streams, precision=PRECISION[dtype]), key
    return _API["api"]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "solve":
        u, dt, dh = _groups(case["npg"], seed, case["scheme"])
        u = u.to(FLOAT[case["dtype"]])
        new = lambda *s: torch.empty((case["npg"],) + s, dtype=u.dtype, device=DEV)  # noqa: E731
        return {"kind": kind, "u": u, "dt": dt, "dh": dh, "kw": dict(
            scheme=case["scheme"], rsolver=case["rsolver"], limiter=case["limiter"], store_flux=case["flux"],
            out=new(5, 16, 16, 16), flux=new(9, 5, 16, 16) if case["flux"] else None, dt_patch=new(8) if case["dt"] else None)}
    if kind == "batch":
        u, dtdh = _levels(case, seed)
        u = u.to(FLOAT[case["dtype"]])
        n = u.shape[0]
        return {"kind": kind, "u": u, "dtdh": dtdh, "kw": dict(
            out=torch.empty((n, 5, 16, 16, 16), dtype=u.dtype, device=DEV),
            flux=torch.empty((n, 9, 5, 16, 16), dtype=u.dtype, device=DEV),
            queue_counter=torch.zeros(1, dtype=torch.int32, device=DEV), groups_per_cu=2)}
    if kind == "uniform":
        cons = _smooth([16 * case[k] for k in ("gz", "gy", "gx")], seed, noise=0.2)
        dh = 1.0 / cons.shape[3]
        dt = _cfl_dt(cons, dh, 0.3)
        return {"kind": kind, "dt": dt, "level": hydro.UniformLevel(cons.to(FLOAT[case["dtype"]]), dh, scheme=case["scheme"])}
    if kind == "twolevel":
        base, fine, dt, dh, lo, m = _two_level(case, seed)
        fathers = [(lo[2] // 8 + i, lo[1] // 8 + j, lo[0] // 8 + k) for k in range(m[0] // 8) for j in range(m[1] // 8)
                   for i in range(m[2] // 8)]
        tab = amr.build_two_level_tables((case["nx"], case["ny"], case["nz"]), fathers)
        t = FLOAT[case["dtype"]]
        # refined patch groups are 16^3 blocks of the refined box in the fathers' order; each holds 8 patches by LocalID
        f = fine.reshape(5, m[0] // 8, 2, 8, m[1] // 8, 2, 8, m[2] // 8, 2, 8).permute(1, 4, 7, 2, 5, 8, 0, 3, 6, 9)
        f = f.reshape(-1, 8, 5, 8, 8, 8)[:, [4 * c + 2 * b + a for a, b, c in amr.LOCAL_XYZ]].reshape(-1, 5, 8, 8, 8)
        lv = amr.TwoLevel(torch, amr.patches_from_grid(base).to(t).contiguous(), f.to(t).contiguous(), tab, dh)
        return {"kind": kind, "dt": dt, "level": lv}
    if kind in ("adjoint", "tangent"):
        u, dt, dh = _groups(case["npg"], seed, sod=False)
        g = torch.Generator(device=DEV).manual_seed(seed + 1)
        v = torch.randn((case["npg"], 5) + ((16,) * 3 if kind == "adjoint" else (22,) * 3), generator=g, dtype=torch.float64, device=DEV)
        return {"kind": kind, "u": u, "v": v, "dt": dt, "dh": dh, "kw": dict(
            rsolver=case["rsolver"], workspace=hydro.adjoint_workspace(case["npg"], DEV))}
    if kind == "rollout":
        cons = _smooth([16 * case[k] for k in ("gz", "gy", "gx")], seed)
        dh = 1.0 / cons.shape[3]
        g = torch.Generator(device=DEV).manual_seed(seed + 1)
        target = 1.0 + 0.1 * torch.randn(cons.shape[1:], generator=g, dtype=torch.float64, device=DEV)
        return {"kind": kind, "level": cons, "target": target, "dt": _cfl_dt(cons, dh, 0.4), "dh": dh, "steps": case["steps"]}
    u, dt, dh = _groups(case["npg"], seed)
    t = FLOAT[case["dtype"]]
    pinned = lambda *s: torch.empty((case["npg"],) + s, dtype=t, pin_memory=True)  # noqa: E731
    h_in = pinned(5, 22, 22, 22)
    h_in.copy_(u)
    _host_api(case["npg"], case["dtype"], case["streams"])
    return {"kind": kind, "key": (case["npg"], case["dtype"], case["streams"]), "in": h_in, "out": pinned(5, 16, 16, 16),
            "flux": pinned(9, 5, 16, 16), "args": hydro.make_args(case["npg"], dt, dh, precision=PRECISION[case["dtype"]])}


def run(s):
    kind = s["kind"]
    if kind == "solve":
        out, flux = hydro.fluid_solver(s["u"], s["dt"], s["dh"], **s["kw"])
        return {"out": out, "flux": flux, "dt": s["kw"]["dt_patch"]}
    if kind == "batch":
        out, flux = hydro.solve_batch(s["u"], s["dtdh"], **s["kw"])
        return {"out": out, "flux": flux}
    if kind == "uniform":
        dt = s["level"].step(s["dt"])
        return {"level": s["level"].level, "dt": dt}
    if kind == "twolevel":
        s["level"].step(s["dt"])
        return {"base": s["level"].base, "fine": s["level"].fine}
    if kind == "adjoint":
        return {"lam_in": hydro.mhm_adjoint(s["u"], s["v"], s["dt"], s["dh"], **s["kw"])}
    if kind == "tangent":
        out, jv = hydro.mhm_tangent(s["u"], s["v"], s["dt"], s["dh"], **s["kw"])
        return {"out": out, "jv": jv}
    if kind == "rollout":
        level = s["level"].detach().requires_grad_(True)
        final = diff.rollout(level, s["steps"], s["dt"], s["dh"])
        loss = diff.density_loss(final, s["target"])
        loss.backward()
        return {"final": final.detach(), "loss": loss.detach(), "grad": level.grad}
    api = _host_api(*s["key"])
    rc = hydro.lib().hydro_asyn_fluid_solver(s["in"].data_ptr(), s["out"].data_ptr(), s["flux"].data_ptr(),
                                             ctypes.byref(s["args"]), s["key"][2])
    if rc != 0:
        raise RuntimeError("hydro_asyn_fluid_solver: %d" % rc)
    api.synchronize()
    return {"out": s["out"], "flux": s["flux"]}


# ---------------------------------------------------------------- what a pass cannot do without

#: Operations per updated cell: three half-step interface solves (75 each), the half-step cell (45), 15 reconstructed face
#: pairs (11 each), three full-step solves with their two states (105 each), the update with its check (45).
CELL_FLOPS = 3 * 75 + 45 + 15 * 11 + 3 * 105 + 45


def work(case):
    kind = case["kind"]
    e = 4 if case.get("dtype") == "f32" else 8
    out, flux = 5 * 16 ** 3, 45 * 16 ** 2
    if kind in ("solve", "host"):
        n = 16 + 2 * _ghost(case.get("scheme", "MHM_RP"))
        b = e * (5 * n ** 3 + out + (flux if case.get("flux", True) else 0) + (8 if case.get("dt") else 0))
        return {"bytes": case["npg"] * b, "flops": case["npg"] * 4096 * CELL_FLOPS}
    if kind == "batch":
        n = case["n0"] + case["n1"] + case["n2"]
        return {"bytes": n * (e * (5 * 22 ** 3 + out + flux) + 16), "flops": n * 4096 * CELL_FLOPS}
    if kind == "uniform":
        n = case["gx"] * case["gy"] * case["gz"]
        return {"bytes": 2 * e * n * out, "flops": n * 4096 * CELL_FLOPS}
    if kind == "twolevel":
        base, fine = 512 * case["nx"] * case["ny"] * case["nz"], 4096 * case["mx"] * case["my"] * case["mz"]
        return {"bytes": 2 * e * 5 * (base + 2 * fine), "flops": (base + 2 * fine) * CELL_FLOPS}
    if kind in ("adjoint", "tangent"):
        b = 8 * (2 * 5 * 22 ** 3 + (1 if kind == "adjoint" else 2) * out)
        return {"bytes": case["npg"] * b, "flops": case["npg"] * 4096 * CELL_FLOPS * (3 if kind == "adjoint" else 2)}
    n = case["gx"] * case["gy"] * case["gz"]
    return {"bytes": case["steps"] * 4 * 8 * n * out, "flops": case["steps"] * n * 4096 * CELL_FLOPS * 4}


# ---------------------------------------------------------------- the same in plain 64-bit torch

def _pressure(c):
    return (GAMMA - 1.0) * (c[4] - 0.5 * (c[1] ** 2 + c[2] ** 2 + c[3] ** 2) / c[0])


def _prim(c):
    """Conserved -> (rho, vx, vy, vz, P), fields first."""
    return [c[0], c[1] / c[0], c[2] / c[0], c[3] / c[0], torch.clamp(_pressure(c), min=0.0)]


def _flux(c, w, d):
    v = w[1 + d]
    f = [v * q for q in c]
    f[1 + d] = f[1 + d] + w[4]
    f[4] = f[4] + v * w[4]
    return f


def _solver(wl, wr, d, rsolver):
    """Interface flux across a d-normal face between primitive states (lists of 5 tensors)."""
    cons = lambda w: [w[0], w[0] * w[1], w[0] * w[2], w[0] * w[3],  # noqa: E731
                      w[4] / (GAMMA - 1.0) + 0.5 * w[0] * (w[1] ** 2 + w[2] ** 2 + w[3] ** 2)]
    ul, ur = cons(wl), cons(wr)
    cl, cr = torch.sqrt(GAMMA * wl[4] / wl[0]), torch.sqrt(GAMMA * wr[4] / wr[0])
    vl, vr = wl[1 + d], wr[1 + d]
    fl, fr = _flux(ul, wl, d), _flux(ur, wr, d)
    if rsolver == "ROE":
        n, t1, t2 = 1 + d, 1 + (d + 1) % 3, 1 + (d + 2) % 3
        sl, sr = torch.sqrt(wl[0]), torch.sqrt(wr[0])
        mean = lambda a, b: (sl * a + sr * b) / (sl + sr)  # noqa: E731
        u, v, w = (mean(wl[k], wr[k]) for k in (n, t1, t2))
        h = mean((ul[4] + wl[4]) / wl[0], (ur[4] + wr[4]) / wr[0])
        q2 = u * u + v * v + w * w
        a = torch.sqrt((GAMMA - 1.0) * (h - 0.5 * q2))
        j = [ur[k] - ul[k] for k in (0, n, t1, t2, 4)]
        a2, a3 = j[2] - v * j[0], j[3] - w * j[0]
        a1 = (GAMMA - 1.0) / (a * a) * (j[0] * (h - u * u) + u * j[1] - j[4] + v * a2 + w * a3)
        a0 = (j[0] * (u + a) - j[1] - a * a1) / (2.0 * a)
        a4 = j[0] - a0 - a1
        d0, d1, d4 = a0 * (u - a).abs(), a1 * u.abs(), a4 * (u + a).abs()
        e2, e3 = a2 * u.abs(), a3 * u.abs()
        diss = {0: d0 + d1 + d4, n: d0 * (u - a) + d1 * u + d4 * (u + a), t1: (d0 + d1 + d4) * v + e2,
                t2: (d0 + d1 + d4) * w + e3, 4: d0 * (h - u * a) + d1 * 0.5 * q2 + e2 * v + e3 * w + d4 * (h + u * a)}
        # an intermediate state without density or pressure takes the HLLE flux instead
        def empty(q):
            return (q[0] <= 0) | (q[4] - 0.5 * (q[1] ** 2 + q[2] ** 2 + q[3] ** 2) / q[0] <= 0)
        one = [ul[k] + a0 * x for k, x in ((0, 1.0), (n, u - a), (t1, v), (t2, w), (4, h - u * a))]
        two = [one[0] + a1, one[1] + a1 * u, one[2] + a1 * v + a2, one[3] + a1 * w + a3, one[4] + a1 * 0.5 * q2 + a2 * v + a3 * w]
        bad = empty(one) | empty(two)
        hlle = _solver(wl, wr, d, "HLLE")
        mid = [torch.where(bad, hlle[k], 0.5 * (fl[k] + fr[k] - diss[k])) for k in range(5)]
        return [torch.where(u - a >= 0, fl[k], torch.where(u + a <= 0, fr[k], mid[k])) for k in range(5)]
    s1, s2 = torch.minimum(vl - cl, vr - cr), torch.maximum(vl + cl, vr + cr)
    zero = torch.zeros_like(s1)
    if rsolver == "HLLE":
        s1, s2 = torch.minimum(s1, zero), torch.maximum(s2, zero)
        return [(s2 * fl[k] - s1 * fr[k] + s1 * s2 * (ur[k] - ul[k])) / (s2 - s1) for k in range(5)]
    ml, mr = wl[0] * (vl - s1), wr[0] * (s2 - vr)
    ss = (wl[4] - wr[4] + ml * vl + mr * vr) / (ml + mr)
    ps = torch.clamp((ml * wr[4] + mr * wl[4] + ml * mr * (vl - vr)) / (ml + mr), min=0.0)
    left = ss >= 0
    pick = lambda a, b: torch.where(left, a, b)  # noqa: E731
    sk, vk, pk = pick(torch.minimum(s1, zero), torch.maximum(s2, zero)), pick(vl, vr), pick(wl[4], wr[4])
    uk = [pick(a, b) for a, b in zip(ul, ur)]
    # F + s (U* - U), U* the state of the contact's side; s = 0 leaves the physical flux
    f = []
    den = ss - sk
    one = den == 0.0
    t = 1.0 / torch.where(one, torch.ones_like(den), den)
    cf, cp = torch.where(one, torch.ones_like(den), t * ss), torch.where(one, torch.zeros_like(den), -t * sk * ps)
    for k in range(5):
        q = (vk - sk) * uk[k]
        q = q + pk if k == 1 + d else q + vk * pk if k == 4 else q
        f.append(cf * q + (cp if k == 1 + d else cp * ss if k == 4 else 0.0))
    return f


def _faces(a, b, c, limiter):
    """Low and high face values of the cells b with neighbours a and c (PLM, MinMod coefficient 1.5)."""
    sl, sr = b - a, c - b
    same = sl * sr > 0
    t = torch.where(same, sl + sr, torch.ones_like(sl))
    vanleer = 2.0 * sl * sr / t
    if limiter == "VANLEER":
        s = vanleer
    else:
        m = torch.minimum(torch.minimum(1.5 * sl.abs(), 1.5 * sr.abs()), 0.5 * (sl + sr).abs())
        if limiter == "VL_GMINMOD":
            m = torch.minimum(m, vanleer.abs())
        s = torch.where(t < 0, -m, m)
    s = torch.where(same, s, torch.zeros_like(s))
    lo = torch.minimum(torch.maximum(b - 0.5 * s, torch.minimum(a, b)), torch.maximum(a, b))
    hi = torch.minimum(torch.maximum(2.0 * b - lo, torch.minimum(b, c)), torch.maximum(b, c))
    return 2.0 * b - hi, hi


def _at(x, d, lo, n):
    """n planes of x from lo along direction d (0 = x, the last axis)."""
    return x.narrow(-1 - d, lo, n)


def _core(x, d, lo, n=16):
    """n planes from lo along the two directions other than d."""
    for k in range(3):
        if k != d:
            x = _at(x, k, lo, n)
    return x


def _hancock(w, k, limiter):
    """Face states (low, high per direction, primitive) of the 18^3 cells of 20^3 primitive inputs after the half step."""
    inner = lambda q, s: [_at(_core(f, s[0], 1, 18), s[0], 1 + s[1], 18) for f in q]  # noqa: E731
    mid = inner(w, (0, 0))
    faces = []
    for d in range(3):
        lo, hi = zip(*(_faces(a, b, c, limiter) for a, b, c in zip(inner(w, (d, -1)), mid, inner(w, (d, 1)))))
        faces += [list(lo), list(hi)]
    cons = [[f[0], f[0] * f[1], f[0] * f[2], f[0] * f[3], f[4] / (GAMMA - 1.0) + 0.5 * f[0] * (f[1] ** 2 + f[2] ** 2 + f[3] ** 2)]
            for f in faces]
    fl = [_flux(c, f, i // 2) for i, (c, f) in enumerate(zip(cons, faces))]
    dif = [sum(fl[2 * d + 1][v] - fl[2 * d][v] for d in range(3)) for v in range(5)]
    return [_prim([c[v] - k * dif[v] for v in range(5)]) for c in cons]


def _step(u, k, scheme="MHM_RP", rsolver="HLLC", limiter="VL_GMINMOD"):
    """One solver call on (n, 5, N, N, N) float64 inputs, k = dt/dh (a number or (n, 1, 1, 1)): (out, flux planes)."""
    c = list(u.unbind(1))
    w = _prim(c)
    g = _ghost(scheme)
    if scheme == "MHM_RP":
        dif = 0.0
        for d in range(3):
            q = [_core(f, d, 1, 20) for f in w]
            f = _solver([_at(x, d, 0, 21) for x in q], [_at(x, d, 1, 21) for x in q], d, rsolver)
            dif = [(_at(x, d, 1, 20) - _at(x, d, 0, 20)) + (0.0 if d == 0 else y) for x, y in zip(f, [0.0] * 5 if d == 0 else dif)]
        half = _prim([_at(_core(x, 0, 1, 20), 0, 1, 20) - 0.5 * k * y for x, y in zip(c, dif)])
    else:
        han = _hancock(w, 0.5 * k, limiter)
    total, planes = 0.0, []
    for d in range(3):
        if scheme == "MHM_RP":
            q = [_core(f, d, 2) for f in half]
            lo, hi = zip(*(_faces(_at(x, d, 0, 18), _at(x, d, 1, 18), _at(x, d, 2, 18), limiter) for x in q))
        else:
            lo, hi = ([_core(f, d, 1) for f in han[2 * d + s]] for s in (0, 1))
        f = _solver([_at(x, d, 0, 17) for x in hi], [_at(x, d, 1, 17) for x in lo], d, rsolver)
        f = torch.stack(f, 1)
        planes += [_at(f, d, p, 1).squeeze(-1 - d) for p in (0, 8, 16)]
        total = total + (_at(f, d, 1, 16) - _at(f, d, 0, 16))
    kk = k.unsqueeze(1) if torch.is_tensor(k) else k
    return _at(_core(u, 0, g), 0, g, 16) - kk * total, torch.stack(planes, 1)


def _steps(u, k, **kw):
    """_step in chunks of patch groups."""
    got = []
    for i in range(0, u.shape[0], 256):
        got.append(_step(u[i:i + 256].double(), k[i:i + 256] if torch.is_tensor(k) else k, **kw))
    return torch.cat([a for a, _ in got]), torch.cat([b for _, b in got])


def _patch_dt(out, dh, safety=0.5):
    s = _signal_speed(out.transpose(0, 1))
    return safety * dh / s.reshape(-1, 2, 8, 2, 8, 2, 8).amax((2, 4, 6)).reshape(-1, 8)


def _join(blocks, shape):
    gz, gy, gx = (n // 16 for n in shape)
    return blocks.reshape(gz, gy, gx, 5, 16, 16, 16).permute(3, 0, 4, 1, 5, 2, 6).reshape(5, *shape)


def _interpolate(c):
    """Conservative quadratic 2x refinement of (5, z, y, x), monotonic with coefficient 2; one cell less on each side."""
    for axis in (3, 2, 1):
        n = c.shape[axis] - 2
        a, b, e = c.narrow(axis, 0, n), c.narrow(axis, 1, n), c.narrow(axis, 2, n)
        s, l, r = 0.125 * (e - a), 0.25 * (b - a), 0.25 * (e - b)
        lim = torch.minimum(torch.where(l.abs() < r.abs(), 2.0 * l.abs(), l.abs()), torch.where(l.abs() < r.abs(), r.abs(), 2.0 * r.abs()))
        s = torch.where(l * r > 0, torch.sign(l) * torch.minimum(s.abs(), lim), 0.0)
        c = torch.stack([b - s, b + s], axis + 1).flatten(axis, axis + 1)
    return c


def _exact_two_level(case, seed):
    base, fine, dt, dh, lo, m = _two_level(case, seed)
    t = FLOAT[case["dtype"]]
    base, fine = base.to(t).double(), fine.to(t).double()
    shape, fshape = base.shape[1:], fine.shape[1:]
    old = base
    out, flux = _steps(_cut(base, 3), dt / dh)
    base = _join(out, shape).clone()
    box = tuple(slice(a, a + b) for a, b in zip(lo, m))
    # register of each face of the box: dt * base flux minus the refined fluxes; patch-group flux planes back to faces
    gz, gy, gx = (n // 16 for n in shape)
    fl = flux.reshape(gz, gy, gx, 9, 5, 16, 16)
    reg = {}
    for d in range(3):                       # 0 = x
        ax = 3 - d                           # axis of (5, z, y, x)
        tang = [b for i, b in enumerate(box) if i != ax - 1]
        for side in (0, 1):
            at = lo[ax - 1] + side * m[ax - 1]
            q, p = divmod(at % shape[ax - 1], 16)
            f = fl.select(ax - 1, q)[:, :, 3 * d + p // 8]                     # (ga, gb, 5, 16, 16)
            f = f.permute(2, 0, 3, 1, 4).flatten(3, 4).flatten(1, 2)
            reg[d, side] = dt * f[:, tang[0], tang[1]]
    for sub in range(2):
        coarse = old if sub == 0 else 0.5 * (old + base)
        c = coarse
        for i in range(3):
            c = c.index_select(i + 1, torch.arange(lo[i] - 3, lo[i] + m[i] + 3, device=DEV) % shape[i])
        w = _interpolate(c)[:, 1:-1, 1:-1, 1:-1].contiguous()
        w[:, 3:-3, 3:-3, 3:-3] = fine
        blk = w.unfold(1, 22, 16).unfold(2, 22, 16).unfold(3, 22, 16).permute(1, 2, 3, 0, 4, 5, 6).reshape(-1, 5, 22, 22, 22)
        out, flux = _steps(blk, dt / dh)
        fine = _join(out, fshape)
        fl = flux.reshape(*(n // 8 for n in m), 9, 5, 16, 16)
        for (d, side) in reg:
            f = fl.select(2 - d, (m[2 - d] // 8 - 1) * side)[:, :, 3 * d + 2 * side]
            f = f.permute(2, 0, 3, 1, 4).flatten(3, 4).flatten(1, 2)
            f = f.reshape(5, f.shape[1] // 2, 2, f.shape[2] // 2, 2).sum((2, 4))
            reg[d, side] = reg[d, side] - 0.125 * dt * f
    base[(slice(None),) + box] = fine.reshape(5, m[0], 2, m[1], 2, m[2], 2).mean((2, 4, 6))
    for (d, side), r in reg.items():
        i = 2 - d
        at = (lo[i] - 1 if side == 0 else lo[i] + m[i]) % shape[i]
        tang = [b for k, b in enumerate(box) if k != i]
        base.select(i + 1, at)[:, tang[0], tang[1]] += (1.0 if side == 0 else -1.0) / dh * r
    f = fine.reshape(5, m[0] // 8, 2, 8, m[1] // 8, 2, 8, m[2] // 8, 2, 8).permute(1, 4, 7, 2, 5, 8, 0, 3, 6, 9)
    f = f.reshape(-1, 8, 5, 8, 8, 8)[:, [4 * c + 2 * b + a for a, b, c in amr.LOCAL_XYZ]].reshape(-1, 5, 8, 8, 8)
    return {"base": amr.patches_from_grid(base), "fine": f}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("solve", "host"):
        scheme = case.get("scheme", "MHM_RP")
        u, dt, dh = _groups(case["npg"], seed, scheme)
        out, flux = _steps(u.to(FLOAT[case["dtype"]]), dt / dh, scheme=scheme, rsolver=case.get("rsolver", "HLLC"),
                           limiter=case.get("limiter", "VL_GMINMOD"))
        if kind == "host":
            return {"out": out, "flux": flux}
        return {"out": out, "flux": flux if case["flux"] else None, "dt": _patch_dt(out, dh) if case["dt"] else None}
    if kind == "batch":
        u, dtdh = _levels(case, seed)
        out, flux = _steps(u.to(FLOAT[case["dtype"]]), (dtdh[:, 0] / dtdh[:, 1]).reshape(-1, 1, 1, 1))
        return {"out": out, "flux": flux}
    if kind == "uniform":
        cons = _smooth([16 * case[k] for k in ("gz", "gy", "gx")], seed, noise=0.2)
        dh = 1.0 / cons.shape[3]
        dt = _cfl_dt(cons, dh, 0.3)
        u = cons.to(FLOAT[case["dtype"]]).double()
        out, _ = _steps(_cut(u, _ghost(case["scheme"])), dt / dh, scheme=case["scheme"])
        return {"level": _join(out, cons.shape[1:]), "dt": _patch_dt(out, dh).min()}
    if kind == "twolevel":
        return _exact_two_level(case, seed)
    if kind in ("adjoint", "tangent"):
        s = prepare(case, seed)
        k, kw, got = s["dt"] / s["dh"], dict(rsolver=case["rsolver"]), []
        for i in range(0, case["npg"], 64):
            u, v = s["u"][i:i + 64], s["v"][i:i + 64]
            if kind == "adjoint":
                u = u.clone().requires_grad_(True)
                got.append((torch.autograd.grad(_step(u, k, **kw)[0], u, v)[0],))
            else:
                got.append(torch.func.jvp(lambda x: _step(x, k, **kw)[0], (u,), (v,)))
        if kind == "adjoint":
            return {"lam_in": torch.cat([g[0] for g in got])}
        return {"out": torch.cat([g[0] for g in got]), "jv": torch.cat([g[1] for g in got])}
    s = prepare(case, seed)
    level = s["level"].detach().requires_grad_(True)
    u, k, shape = level, s["dt"] / s["dh"], level.shape[1:]
    for _ in range(s["steps"]):
        u = _join(_step(_cut(u, 3), k)[0], shape)
    loss = ((u[0] - s["target"]) ** 2).sum()
    loss.backward()
    return {"final": u.detach(), "loss": loss.detach(), "grad": level.grad}
