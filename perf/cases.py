"""Work that programs give this library, as measurable cases.

Each case is one call (or one time step's worth of calls) through a public
entry point: the reference-mode solvers behind the plugin interface, the
Jacobi-scaled and multigrid PCG of a resident system in either precision, a
projection step with a new density, a batch and a served stream.  Every system
is a periodic two-phase pressure system as in aphros_amd/synth.py: spheres of
density 1 in a fluid of density `ratio`, harmonic face densities, the
projection's sign.  The right-hand side is close to the benchmark systems'
white noise, but it is the operator applied in FP64 to a given pressure, so the
solution that a solve approaches is known.
"""
import ctypes as C
import math
import random

import numpy as np
import torch

from aphros_amd import _lib as L
from aphros_amd.batch import Batch
from aphros_amd.linear import MakeLinearSolver, Mesh, Vars
from aphros_amd.serve import Server
from aphros_amd.solver import Poisson

# Relative residual of the solves: small enough that the solution, and not
# the point at which an iteration happens to stop, is what two runs compare.
TOL = 1e-11


def listed():
    return [
        # the plugin as the reference's time loop calls it: one 32^3 block
        # (the reference's linear test) with halos in host memory, the
        # module's defaults (reference-mode CG), two time steps whose
        # densities differ
        dict(name="plugin_cg_32", kind="plugin", nx=32, ny=32, nz=32, spheres=4, rmin=0.08,
             rmax=0.2, ratio=10.0, steps=2),
        # reference-mode Jacobi for callers that cannot allocate: a ragged
        # block, a fixed number of sweeps
        dict(name="jacobi_noalloc_ragged", kind="jacobi", nx=60, ny=45, nz=52, spheres=8,
             rmin=0.08, rmax=0.15, ratio=1000.0, sweeps=400),
        # reference-mode CG on the 64^3 benchmark geometry, resident system
        dict(name="cg_64", kind="cg", nx=64, ny=64, nz=64, spheres=8, rmin=0.08, rmax=0.15,
             ratio=1000.0),
        # Jacobi-scaled PCG, mixed precision, odd edges (nothing coarsens),
        # with a mass term (an implicit diffusion step)
        dict(name="pcg_mixed_odd", kind="pcg", nx=101, ny=75, nz=93, spheres=8, rmin=0.08,
             rmax=0.15, ratio=100.0, precision="mixed", precond="jacobi", mass=0.05),
        # the plain FP64 form, Jacobi-scaled, as the drop-in's streaming solver
        dict(name="pcg_fp64_128", kind="pcg", nx=128, ny=128, nz=128, spheres=32, rmin=0.08,
             rmax=0.15, ratio=1000.0, precision="fp64", precond="jacobi", mass=0.0),
        # multigrid, mixed precision: a small resident system, where launches
        # and latency count
        dict(name="mg_mixed_64", kind="pcg", nx=64, ny=64, nz=64, spheres=8, rmin=0.08,
             rmax=0.15, ratio=1000.0, precision="mixed", precond="mg", mass=0.0),
        # one projection step: the system assembled from a new density, the
        # solve from the last step's pressure, the corrected fluxes
        dict(name="step_mg_128x96x160", kind="step", nx=128, ny=96, nz=160, spheres=16,
             rmin=0.05, rmax=0.15, ratio=1000.0),
        # multigrid in FP64, the baseline form of the mixed one
        dict(name="mg_fp64_192", kind="pcg", nx=192, ny=192, nz=192, spheres=16, rmin=0.05,
             rmax=0.15, ratio=1000.0, precision="fp64", precond="mg", mass=0.0),
        # the 256^3 and 512^3 benchmark geometries, mixed precision
        dict(name="mg_mixed_256", kind="pcg", nx=256, ny=256, nz=256, spheres=32, rmin=0.08,
             rmax=0.15, ratio=1000.0, precision="mixed", precond="mg", mass=0.0),
        dict(name="mg_mixed_512", kind="pcg", nx=512, ny=512, nz=512, spheres=128, rmin=0.02,
             rmax=0.06, ratio=1000.0, precision="mixed", precond="mg", mass=0.0),
        # many uneven systems at once: new right-hand sides in, solutions out
        dict(name="batch_12", kind="batch", systems=12, emin=32, emax=128),
        # a served burst: requests of mixed sizes, each a sequence of
        # warm-started correlated right-hand sides
        dict(name="served_5", kind="served", requests=5, steps=3, emin=48, emax=128),
    ]


def _even_log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["plugin", "jacobi", "cg", "pcg_j", "pcg_j", "mg", "mg", "mg", "mg_fp64",
                       "step", "step", "batch", "served"])
    geo = dict(spheres=rng.randint(2, 32), rmin=0.05, rmax=0.15,
               ratio=10.0 ** rng.uniform(1.0, 3.0))

    def edges(lo, hi, cells, mult=1):
        """Three edges (multiples of `mult`) of a block of about `cells`."""
        c = _even_log(rng, *cells) ** (1 / 3)
        e = [c * math.exp(rng.uniform(-0.3, 0.3)) for _ in range(3)]
        return dict(zip(("nx", "ny", "nz"),
                        (int(min(hi, max(lo, mult * round(v / mult)))) for v in e)))

    if kind == "plugin":
        return dict(kind="plugin", **edges(8, 48, (12 ** 3, 36 ** 3)), **geo, steps=2)
    if kind == "jacobi":
        return dict(kind="jacobi", **edges(8, 128, (16 ** 3, 96 ** 3)), **geo,
                    sweeps=rng.randint(50, 500))
    if kind == "cg":
        return dict(kind="cg", **edges(8, 80, (16 ** 3, 56 ** 3)), **geo)
    if kind == "pcg_j":
        return dict(kind="pcg", **edges(16, 160, (24 ** 3, 112 ** 3)), **geo,
                    precision=rng.choice(["mixed", "fp64"]), precond="jacobi",
                    mass=rng.choice([0.0, 0.05]))
    if kind == "mg":
        big = rng.random() < 0.4
        e = edges(160, 448, (192 ** 3, 400 ** 3), 32) if big else \
            edges(32, 224, (40 ** 3, 180 ** 3), 16)
        return dict(kind="pcg", **e, **geo, precision="mixed", precond="mg",
                    mass=rng.choice([0.0, 0.0, 0.05]))
    if kind == "mg_fp64":
        return dict(kind="pcg", **edges(32, 256, (48 ** 3, 200 ** 3), 16), **geo,
                    precision="fp64", precond="mg", mass=0.0)
    if kind == "step":
        return dict(kind="step", **edges(32, 288, (48 ** 3, 256 ** 3), 16), **geo)
    if kind == "batch":
        return dict(kind="batch", systems=rng.randint(4, 12), emin=32, emax=128)
    return dict(kind="served", requests=rng.randint(2, 5), steps=rng.randint(2, 3), emin=48,
                emax=128)


# ------------------------------------------------------------------ inputs

def _density(case, seed):
    """Cell density (nz, ny, nx) on the GPU: periodic spheres of density 1 in
    a box whose longest edge is 1 (cubic cells)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    h = 1.0 / max(nx, ny, nz)
    rng = random.Random(seed)
    axes = [(torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) * h for n in (nx, ny, nz)]
    ext = [n * h for n in (nx, ny, nz)]
    inside = torch.zeros((nz, ny, nx), dtype=torch.bool, device="cuda")
    for _ in range(case["spheres"]):
        r = rng.uniform(case["rmin"], case["rmax"])
        d2 = []
        for a, e in zip(axes, ext):
            d = (a - rng.uniform(0.0, e)).abs()
            d2.append(torch.minimum(d, e - d) ** 2)
        near = [(d < r * r).nonzero().flatten() for d in d2]
        if min(v.numel() for v in near) == 0:
            continue
        ix, iy, iz = near
        ball = d2[2][iz][:, None, None] + d2[1][iy][None, :, None] + d2[0][ix][None, None, :] \
            < r * r
        sub = torch.index_select(inside, 0, iz)
        sub[:, iy[:, None], ix[None, :]] |= ball
        inside[iz] = sub
    rho = torch.full((nz, ny, nx), float(case["ratio"]), dtype=torch.float64, device="cuda")
    rho[inside] = 1.0
    return rho, h


def _faces(rho, h):
    """Minus the coupling of each cell's lower x, y and z face: h / rho_f with
    the harmonic face density."""
    inv = 1.0 / rho
    return [(0.5 * (inv + inv.roll(1, a))) * h for a in (2, 1, 0)]


def _apply(k, mass, x):
    """A x of the assembled system, in FP64, as a sum of face differences."""
    out = mass * x if mass else torch.zeros_like(x)
    for kf, a in zip(k, (2, 1, 0)):
        flux = kf * (x - x.roll(1, a))
        out += flux
        out -= flux.roll(-1, a)
    return out


def _pressure(k, mass, seed):
    """A pressure (nz, ny, nx), FP64, unit RMS and (without a mass term) zero
    mean, whose right-hand side A x is close to white noise: some conjugate
    gradients on noise, preconditioned by the Fourier inverse of the operator
    with the conductances' median.  What is left of its residual only means
    that A x is not quite that noise."""
    shape = k[0].shape
    nz, ny, nx = shape
    g = torch.Generator(device="cuda").manual_seed(seed)
    f = torch.rand(shape, generator=g, device="cuda", dtype=torch.float64) - 0.5
    f -= f.mean()
    s = [4.0 * torch.sin(math.pi * v) ** 2
         for v in (torch.fft.fftfreq(nz, device="cuda", dtype=torch.float64),
                   torch.fft.fftfreq(ny, device="cuda", dtype=torch.float64),
                   torch.fft.rfftfreq(nx, device="cuda", dtype=torch.float64))]
    inv = s[0][:, None, None] + s[1][None, :, None] + s[2][None, None, :]
    inv = inv * float(k[0].flatten()[::97].median()) + mass
    inv[0, 0, 0] = inv[0, 0, 0] if mass else math.inf
    inv = 1.0 / inv
    x, r, p, rz = torch.zeros_like(f), f, None, 1.0
    for _ in range(24):
        z = torch.fft.irfftn(torch.fft.rfftn(r) * inv, s=shape)
        new = (r * z).sum()
        p = z if p is None else z + (new / rz) * p
        rz = new
        q = _apply(k, mass, p)
        alpha = rz / (p * q).sum()
        x += alpha * p
        r = r - alpha * q
    if not mass:
        x -= x.mean()
    return x / x.square().mean().sqrt()


def _expr(k, mass, b):
    """Dense Expr (nz, ny, nx, 8): the diagonal as the ordered sum of its
    faces, as the projection assembles it."""
    e = torch.empty(tuple(b.shape) + (8,), dtype=torch.float64, device="cuda")
    for d, (kf, a) in enumerate(zip(k, (2, 1, 0))):
        e[..., 1 + 2 * d] = -kf
        e[..., 2 + 2 * d] = -kf.roll(-1, a)
    s = e[..., 1].clone()
    for q in range(2, 7):
        s += e[..., q]
    e[..., 0] = mass - s if mass else -s
    e[..., 7] = -b
    return e


def _operator(case, seed):
    """(face conductances, mass term, cell size) of a case."""
    rho, h = _density(case, seed)
    return _faces(rho, h), case.get("mass", 0.0) * h / case["ratio"], h


def _system(case, seed):
    """(Expr, pressure, cell size) of a case, on the GPU."""
    k, mass, h = _operator(case, seed)
    x = _pressure(k, mass, seed)
    b = _apply(k, mass, x)
    e = _expr(k, mass, b)
    torch.cuda.synchronize()
    return e, x, h


def _ref_tol(e, h):
    """The reference's residual is sqrt(sum r^2 / h^3): a tolerance of TOL on
    the relative residual."""
    return TOL * float(e[..., 7].norm()) / math.sqrt(h ** 3)


def _edge_list(case, count):
    """Edges of the systems of a batch or stream, spread over the case's range."""
    sizes = [v for v in (32, 48, 64, 96, 128) if case["emin"] <= v <= case["emax"]]
    return [sizes[(3 * i + 1) % len(sizes)] for i in range(count)]


def _sub(n, seed):
    """One system of a batch or stream."""
    r = random.Random(seed)
    return dict(nx=n, ny=n, nz=n, spheres=r.randint(1, 16), rmin=0.05, rmax=0.15,
                ratio=10.0 ** r.uniform(1.0, 3.0))


def _step_pressures(k, seed, steps):
    """Pressures of a served sequence: each differs by 1 % from the last."""
    x = [_pressure(k, 0.0, seed)]
    for j in range(1, steps):
        x.append(x[-1] + 0.01 * _pressure(k, 0.0, seed + 7919 * j))
    return x


# ------------------------------------------------------------------ states

def prepare(case, seed):
    kind = case["kind"]
    nx, ny, nz = case.get("nx"), case.get("ny"), case.get("nz")
    if kind == "plugin":
        m = None
        fields = []
        for k in range(case["steps"]):
            e, _, h = _system(case, seed + 7919 * k)
            m = Mesh((nx, ny, nz), h=(h, h, h), hl=2)
            box = m.box()
            fs = np.zeros((box[2], box[1], box[0], 8))
            fs[2:2 + nz, 2:2 + ny, 2:2 + nx] = e.cpu().numpy()
            fields.append(fs)
            tol = _ref_tol(e, h)
        var = Vars(String={"linsolver_symm": "hip"}, Double={"hypre_symm_tol": tol},
                   Int={"hypre_symm_maxiter": 20000})
        return dict(kind=kind, m=m, fields=fields, solver=MakeLinearSolver(var, "symm", m),
                    zero=np.zeros(m.nslots()), sol=[np.zeros(m.nslots()) for _ in fields])
    if kind == "jacobi":
        e, _, h = _system(case, seed)
        d = L.Desc()
        L.lib().aphpois_desc_default(C.byref(d))
        d.nx, d.ny, d.nz, d.h3 = nx, ny, nz, h ** 3
        d.method, d.resmode, d.tol = L.JACOBI, L.RES_L2, 0.0
        d.miniter, d.maxiter = 0, case["sweeps"] - 1
        return dict(kind=kind, desc=d, e=e, x=torch.empty_like(e[..., 0]))
    if kind in ("cg", "pcg"):
        e, x, h = _system(case, seed)
        if kind == "cg":
            s = Poisson((nz, ny, nx), method=L.CONJUGATE, resmode=L.RES_L2, tol=_ref_tol(e, h),
                        miniter=0, maxiter=100000, h3=h ** 3)
        else:
            s = Poisson((nz, ny, nx), method=L.PCG,
                        precision=L.MIXED if case["precision"] == "mixed" else L.FP64,
                        resmode=L.RES_REL_TRUE, tol=TOL, maxiter=100000, h3=h ** 3,
                        precond=L.PRECOND_MG if case["precond"] == "mg" else L.PRECOND_JACOBI)
        s.set_system_device(e.data_ptr())
        out = torch.empty_like(x)
        del e, x
        torch.cuda.empty_cache()
        return dict(kind=kind, solver=s, x=out)
    if kind == "step":
        rho, h = _density(case, seed)
        k = _faces(rho, h)
        p = _pressure(k, 0.0, seed)
        # fluxes before the projection whose divergence is that of the
        # pressure's: -k grad p plus a divergence-free part
        ffv = torch.stack([kf * (p - p.roll(1, a)) for kf, a in zip(k, (2, 1, 0))])
        ffv += torch.tensor([0.3, -0.2, 0.1], dtype=torch.float64,
                            device="cuda").view(3, 1, 1, 1) * h
        old = p + 0.05 * _pressure(k, 0.0, seed + 7919)  # the last step's pressure
        s = Poisson((nz, ny, nx), method=L.PCG, precision=L.MIXED, resmode=L.RES_REL_TRUE,
                    tol=TOL, maxiter=100000, h3=h ** 3, precond=L.PRECOND_MG)
        torch.cuda.synchronize()
        return dict(kind=kind, solver=s, rho=rho, ffv=ffv, old=old, p=torch.empty_like(p),
                    out=torch.empty_like(ffv), h=h)
    if kind == "batch":
        b = Batch(precision=L.MIXED, tol=TOL, precond=L.PRECOND_MG)
        slots = []
        for i, n in enumerate(_edge_list(case, case["systems"])):
            e, _, _ = _system(_sub(n, seed + i), seed + i)
            e7 = e[..., 7].cpu().numpy().copy()
            slots.append((b.add(e.cpu().numpy()), e7, np.zeros((n, n, n))))
        return dict(kind=kind, batch=b, slots=slots)
    srv = Server(precision=L.MIXED, tol=TOL, mem_budget=200 << 30, precond=L.PRECOND_MG)
    reqs = []
    for i, n in enumerate(_edge_list(case, case["requests"])):
        k, _, _ = _operator(_sub(n, seed + i), seed + i)
        b = [_apply(k, 0.0, x) for x in _step_pressures(k, seed + i, case["steps"])]
        reqs.append((_expr(k, 0.0, b[0]).cpu().numpy(), [(-v).cpu().numpy() for v in b]))
    return dict(kind=kind, server=srv, requests=reqs, steps=case["steps"])


def run(state):
    kind = state["kind"]
    if kind == "plugin":
        for fs, sol in zip(state["fields"], state["sol"]):
            state["solver"].Solve(fs, state["zero"], sol, state["m"])
        return list(state["sol"])
    if kind == "jacobi":
        info = L.Info()
        L.check(L.lib().aphpois_solve_device_noalloc(
            C.byref(state["desc"]), state["e"].data_ptr(), None, state["x"].data_ptr(), None,
            C.byref(info)))
        return state["x"]
    if kind in ("cg", "pcg"):
        state["solver"].solve_device(state["x"].data_ptr())
        return state["x"]
    if kind == "step":
        s, h = state["solver"], state["h"]
        rho, ffv, p, out = (state[k].data_ptr() for k in ("rho", "ffv", "p", "out"))
        L.check(L.lib().aphpois_assemble_device(s.h, rho, ffv, None, h, 1.0, 1))
        s.solve_device(p, state["old"].data_ptr())
        L.check(L.lib().aphpois_flux_correct_device(s.h, p, rho, ffv, out, h, 1.0))
        return {"p": state["p"], "flux": state["out"]}
    if kind == "batch":
        b = state["batch"]
        for slot, e7, zero in state["slots"]:
            b.set_rhs(slot, e7, zero)
        b.solve()
        return [b.get(slot)[0] for slot, _, _ in state["slots"]]
    srv = state["server"]
    ids = [srv.submit(e, nsteps=state["steps"], e7_steps=e7, want_x=True)
           for e, e7 in state["requests"]]
    return [srv.wait(i)["x"] for i in ids]


# ------------------------------------------------------------------ figures

def _cells(case):
    if "nx" in case:
        return case["nx"] * case["ny"] * case["nz"]
    count = case.get("systems") or case["requests"]
    return sum(n ** 3 for n in _edge_list(case, count))


def work(case):
    """Bytes: the system's symmetric coefficients (4 of 8 B) and constant term
    read and the solution written, once.  Flops: an application of the
    operator (13) and three vector updates and products (10) per iteration,
    with the iterations that the method needs at these sizes (a multigrid
    cycle: 6 applications more)."""
    n, kind = _cells(case), case["kind"]
    edge = n ** (1 / 3)
    if kind == "jacobi":
        return {"bytes": 80.0 * n, "flops": 15.0 * n * case["sweeps"]}
    if kind == "plugin":
        return {"bytes": 80.0 * n * case["steps"], "flops": 23.0 * n * 10 * edge * case["steps"]}
    if kind == "cg":
        return {"bytes": 48.0 * n, "flops": 23.0 * n * 50 * edge}
    if kind == "pcg" and case["precond"] == "jacobi":
        return {"bytes": 48.0 * n, "flops": 25.0 * n * 8 * edge}
    if kind == "pcg":
        return {"bytes": 48.0 * n, "flops": 100.0 * n * 40}
    if kind == "step":
        # density, fluxes and the old pressure in; pressure and fluxes out
        return {"bytes": 72.0 * n, "flops": 100.0 * n * 40}
    if kind == "batch":
        return {"bytes": 56.0 * n, "flops": 100.0 * n * 30}
    return {"bytes": (72.0 + 16.0 * case["steps"]) * n, "flops": 100.0 * n * 30 * case["steps"]}


# ------------------------------------------------------------------ exact

def _jacobi_exact(case, seed):
    e, _, _ = _system(case, seed)
    u = torch.zeros_like(e[..., 0])
    c = [e[..., q].contiguous() for q in range(8)]
    for _ in range(case["sweeps"]):
        s = c[7].clone()
        for q, (a, sh) in enumerate(((2, 1), (2, -1), (1, 1), (1, -1), (0, 1), (0, -1))):
            s += u.roll(sh, a) * c[1 + q]
        u = -s / c[0]
    return u


def exact(case, seed):
    kind = case["kind"]
    if kind == "jacobi":
        return _jacobi_exact(case, seed)
    if kind in ("cg", "pcg"):
        k, mass, _ = _operator(case, seed)
        return _pressure(k, mass, seed)
    if kind == "plugin":
        out = []
        for j in range(case["steps"]):
            nx, ny, nz = case["nx"], case["ny"], case["nz"]
            k, mass, _ = _operator(case, seed + 7919 * j)
            x = _pressure(k, mass, seed + 7919 * j).cpu().numpy()
            # the halos that Solve fills periodically
            ix, iy, iz = (np.arange(-2, n + 3) % n for n in (nx, ny, nz))
            out.append(x[np.ix_(iz, iy, ix)].reshape(-1))
        return out
    if kind == "step":
        k, _, h = _operator(case, seed)
        p = _pressure(k, 0.0, seed)
        # the pressure's fluxes cancel: the divergence-free part is left
        flux = torch.tensor([0.3, -0.2, 0.1], dtype=torch.float64, device="cuda") * h
        return {"p": p, "flux": flux.view(3, 1, 1, 1).expand((3,) + tuple(p.shape)).contiguous()}
    out = []
    for i, n in enumerate(_edge_list(case, case.get("systems") or case["requests"])):
        k, _, _ = _operator(_sub(n, seed + i), seed + i)
        out.append(_pressure(k, 0.0, seed + i) if kind == "batch" else
                   _step_pressures(k, seed + i, case["steps"])[-1])
    return out
