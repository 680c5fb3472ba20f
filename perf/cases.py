"""The work a simulation has this framework do, as measurable cases.

A fluid or ferrofluid simulation calls the framework several times in each
substep: it reclassifies its cells, redistances the level set, assembles and
solves the pressure system (and, for a ferrofluid, the magnetic potential; with
capillarity, one system per axis), applies the pressure and extends the
velocity outside the fluid.  A service solves many such systems at once.  Each
kind of case below is one of these calls, through the package's public entry
points, on seeded scenes of the sizes the package's workloads name (2D 128^2,
3D 128^3 and 256^3, batches with sides in [32, 128], requests with sides in
[64, 256]).
"""
import math
import os
import random
import sys
import types

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "taichi-ferrofluid_amd"))

from mgpcg_amd import batch, cells, level_set, mgpcg, projection, serve, systems  # noqa: E402
from mgpcg_amd.magnetic_force import MagneticForceStrategy  # noqa: E402
from mgpcg_amd.potential_function import PotentialFunctionStrategy  # noqa: E402
from mgpcg_amd.pressure_project import PressureProjectStrategy  # noqa: E402
from mgpcg_amd.surface_tension import SurfaceTension  # noqa: E402
from mgpcg_amd.volume_control import PressureProjectWithVolumeControlStrategy  # noqa: E402

DEVICE = "cuda"
FLUID, AIR, SOLID = 0, 1, 2
DT, RHO, P0 = 1.25e-2, 1000.0, 1e-3
SIGMA = 7.28e-2
MU0, MAG_K = 4 * math.pi * 1e-7, 5.0


def listed():
    return [
        # one pressure projection of a 2D simulation: the smallest call, all latency
        {"name": "pressure_2d_128", "kind": "pressure", "n0": 128, "n1": 128, "n2": 0, "L": 4,
         "gfm": False, "precision": "plain", "spheres": 1},
        # the same in 3D with ghost-fluid weights: the ordinary size
        {"name": "pressure_3d_128", "kind": "pressure", "n0": 128, "n1": 128, "n2": 128, "L": 5,
         "gfm": True, "precision": "mixed", "spheres": 1},
        # ... and the largest: a system beyond the last-level cache
        {"name": "pressure_3d_256", "kind": "pressure", "n0": 256, "n1": 256, "n2": 256, "L": 6,
         "gfm": True, "precision": "mixed", "spheres": 8},
        # a service with eight solve requests in flight (the package's headline)
        {"name": "served_8x128", "kind": "served", "count": 8, "lo": 128, "hi": 128, "mix": 1},
        # a batch of uneven systems of all four kinds a substep solves
        {"name": "batch_16_mixed", "kind": "batch", "count": 16, "lo": 32, "hi": 128, "mix": 100},
        # the 2D ferrofluid demo's substep: magnetic potential to its iteration
        # cap, magnetic pressure, and the force applied
        {"name": "ferro_2d_128", "kind": "ferro", "n0": 128, "n1": 128, "n2": 0, "L": 4},
        # a volume-controlled projection on an uneven box: cell types, volume,
        # assembly, solve, pressure applied
        {"name": "volume_3d_uneven", "kind": "volume", "n0": 144, "n1": 96, "n2": 176, "L": 5,
         "precision": "plain"},
        # implicit surface tension: normals, curvature and one system per axis
        {"name": "surface_3d_128", "kind": "surface", "n0": 128, "n1": 128, "n2": 128, "L": 5},
        # the level set made a distance again after advection: 2D demo size,
        # an odd 3D box, the largest 3D grid
        {"name": "redistance_2d_128", "kind": "redistance", "n0": 128, "n1": 128, "n2": 0},
        {"name": "redistance_3d_odd", "kind": "redistance", "n0": 131, "n1": 97, "n2": 150},
        {"name": "redistance_3d_256", "kind": "redistance", "n0": 256, "n1": 256, "n2": 256},
        # the velocity extended ten cells beyond the fluid
        {"name": "extrapolate_3d_128", "kind": "extrapolate", "n0": 128, "n1": 128, "n2": 128},
    ]


def _log_side(rng, lo, hi, step):
    side = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(side / step)) * step))


def _sides(rng, dim, lo, hi, step):
    n = [_log_side(rng, lo, hi, step) for _ in range(dim)]
    return {"n0": n[0], "n1": n[1], "n2": n[2] if dim == 3 else 0}


def draw(rng):
    kind = rng.choice(["pressure", "pressure", "served", "batch", "ferro", "volume", "surface",
                       "redistance", "redistance", "extrapolate", "extrapolate"])
    case = {"kind": kind}
    if kind in ("served", "batch"):
        lo, hi = ((64, 144) if kind == "served" else (32, 112))
        case.update(count=rng.randint(2, 8 if kind == "served" else 12), lo=lo, hi=hi,
                    mix=rng.randrange(1 << 20))
        return case
    dim = rng.choice([2, 3, 3])
    if kind in ("redistance", "extrapolate"):
        case.update(_sides(rng, dim, 32, 1000 if dim == 2 else 200, 1))
        return case
    if kind == "ferro":
        dim = 2
    L = 4
    case.update(_sides(rng, dim, 48, 512 if dim == 2 and kind != "ferro" else 176, 1 << (L - 1)),
                L=L)
    if kind == "pressure":
        case.update(gfm=rng.random() < 0.7, precision=rng.choice(["plain", "mixed", "mixed"]),
                    spheres=rng.randint(1, 6))
    if kind == "volume":
        case.update(precision=rng.choice(["plain", "mixed"]))
    return case


# ---------------------------------------------------------------------------
# scenes, made on the device from a seed
# ---------------------------------------------------------------------------
def _res(case):
    return [case["n0"], case["n1"]] + ([case["n2"]] if case["n2"] else [])


def _centres(res, dx):
    return torch.meshgrid(*[(torch.arange(n, dtype=torch.float64, device=DEVICE) + 0.5) * dx
                            for n in res], indexing="ij")


def _pool(res, seed, spheres):
    """dx and the signed distance to a pool with spheres above and in it."""
    rng = random.Random(seed)
    dx = 1.0 / max(res)
    ext = [n * dx for n in res]
    X = _centres(res, dx)
    phi = X[1] - rng.uniform(0.27, 0.36) * ext[1]
    for _ in range(spheres):
        r = rng.uniform(0.08, 0.16) * min(ext)
        c = [rng.uniform(0.25, 0.75) * e for e in ext]
        d = sum((x - y) ** 2 for x, y in zip(X, c)).sqrt() - r
        phi = torch.minimum(phi, d)
    return dx, phi.to(torch.float32)


def _cell_types(phi, dtype=torch.int32):
    ct = torch.where(phi <= 0, FLUID, AIR).to(dtype)
    for a in range(phi.dim()):
        ct.select(a, 0).fill_(SOLID)
        ct.select(a, phi.shape[a] - 1).fill_(SOLID)
    return ct


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _faces(res, gen, scale=1.0):
    """One field per axis on that axis's faces, uniform in [-scale, scale]."""
    out = []
    for k in range(len(res)):
        shape = [n + (a == k) for a, n in enumerate(res)]
        u = torch.rand(shape, dtype=torch.float32, device=DEVICE, generator=gen)
        out.append((2 * u - 1) * scale)
    return out


def _scene(kind, res, seed, spheres=1, gfm=True, L=5):
    """A system in the form that systems.assemble takes, on the device."""
    dx, phi = _pool(res, seed, spheres)
    gen = _generator(seed)
    out = {"kind": kind, "dim": len(res), "res": list(res), "L": L, "dx": dx, "dt": DT,
           "rho": RHO, "scale_A": DT / (RHO * dx * dx), "scale_b": 1.0 / dx, "p0": P0,
           "gfm": gfm, "c_max": 100.0, "phi": phi, "cell_type": _cell_types(phi),
           "velocity": _faces(res, gen)}
    if kind == "volume":
        out["c"] = random.Random(seed + 1).uniform(-0.5, 0.5)
    if kind == "psi":
        out.update(chi=torch.where(phi <= 0, 2.0, 0.0), H_ext=_faces(res, gen, 1.2e4))
    if kind == "surface":
        out.update(d=seed % len(res), sigma=SIGMA)
    return out


def _box_list(case):
    rng = random.Random(case["mix"])
    return [[_log_side(rng, case["lo"], case["hi"], 16) for _ in range(3)]
            for _ in range(case["count"])]


def _scenes(case, seed):
    kinds = ("psi", "pressure", "surface", "volume") if case["kind"] == "batch" else ("pressure",)
    return [_scene(kinds[i % len(kinds)], res, 1000 * seed + i)
            for i, res in enumerate(_box_list(case))]


def _solver(res, L, precision):
    return mgpcg.MGPCGPoissonSolver(len(res), res, L, 2, 10, precision=precision, device=DEVICE)


def _pressure_strategy(s, cls=PressureProjectStrategy, *more):
    st = cls(s["dim"], s["velocity"], s["gfm"], s["phi"], s["p0"], *more, c_max=s["c_max"])
    st.scale_A, st.scale_b = s["scale_A"], s["scale_b"]
    return st


def _magnet(res, dx, seed):
    """A smooth applied field on the faces: uniform along y plus a gradient."""
    rng = random.Random(seed + 2)
    h0, gr = rng.uniform(8e3, 1.2e4), rng.uniform(2e3, 4e3)
    out = []
    for k in range(len(res)):
        X = torch.meshgrid(*[(torch.arange(n + (a == k), dtype=torch.float64, device=DEVICE)
                              + (0.0 if a == k else 0.5)) * dx for a, n in enumerate(res)],
                           indexing="ij")
        out.append((h0 * (k == 1) + gr * (X[1] if k == 1 else -X[0] * (k == 0)))
                   .to(torch.float32).contiguous())
    return out


def _advected(res, seed):
    """A level set as advection leaves it: the zero crossing of a scene, the
    values no longer distances."""
    dx, phi = _pool(res, seed, 3)
    X = _centres(res, dx)
    wave = 1.0 + 0.4 * torch.sin(9.0 * X[0] + seed % 7) * torch.cos(7.0 * X[-1])
    return dx, (phi.double() * wave).to(torch.float32)


def prepare(case, seed):
    kind = case["kind"]
    st = types.SimpleNamespace(kind=kind)
    if kind == "served":
        st.scenes = _scenes(case, seed)
        st.server = serve.Server(64 << 30, precision="mixed", n_levels=5, device="cuda:0")
        return st
    if kind == "batch":
        st.scenes = _scenes(case, seed)
        st.solvers = [_solver(s["res"], s["L"], "mixed") for s in st.scenes]
        st.batch = batch.BatchSolver()
        return st
    res = _res(case)
    if kind == "redistance":
        dx, st.phi = _advected(res, seed)
        st.ls = level_set.FastSweepingLevelSet(len(res), res, dx, device=DEVICE)
        return st
    if kind == "extrapolate":
        _, phi = _pool(res, seed, 2)
        st.cell_type = _cell_types(phi, torch.int8)
        st.given = _faces(res, _generator(seed))
        st.velocity = [torch.empty_like(u) for u in st.given]
        return st
    if kind == "pressure":
        st.scene = _scene("pressure", res, seed, case["spheres"], case["gfm"], case["L"])
        st.solver = _solver(res, case["L"], case["precision"])
        st.strategy = _pressure_strategy(st.scene)
        return st
    s = st.scene = _scene("pressure", res, seed, 2, True, case["L"])
    st.velocity = [u.clone() for u in s["velocity"]]
    st.given = s["velocity"]
    s["velocity"] = st.velocity
    if kind == "volume":
        s["c_max"] = 1e3
        st.cell_type = torch.empty(res, dtype=torch.int8, device=DEVICE).fill_(AIR)
        cells.init_boundary(st.cell_type)
        st.solver = _solver(res, case["L"], case["precision"])
        ls = level_set.LevelSet(len(res), res, s["dx"], phi=s["phi"], device=DEVICE)
        st.strategy = _pressure_strategy(s, PressureProjectWithVolumeControlStrategy, ls, DT)
        # the target volume, a little above the present one
        st.target = 1.01 * float((s["phi"] <= 0).sum().item())
        return st
    if kind == "surface":
        st.solver = _solver(res, case["L"], "plain")
        sim = types.SimpleNamespace(
            dim=len(res), res=res, dt=DT, dx=s["dx"], real=float, velocity=st.velocity,
            level_set=level_set.LevelSet(len(res), res, s["dx"], phi=s["phi"], device=DEVICE),
            poisson_solver=st.solver, verbose=False)
        st.tension = SurfaceTension(sim, sigma=SIGMA)
        return st
    # ferro
    st.solver = _solver(res, case["L"], "plain")
    st.H = _magnet(res, s["dx"], seed)
    st.chi = torch.where(s["phi"] <= 0, 2.0, 0.0)
    st.cell_type = s["cell_type"].to(torch.int8)
    st.potential = PotentialFunctionStrategy(len(res), res, s["dx"], st.H, st.chi)
    st.strategy = MagneticForceStrategy(len(res), st.velocity, True, s["phi"], s["p0"], MU0,
                                        MAG_K, st.H, c_max=s["c_max"])
    st.strategy.scale_A, st.strategy.scale_b = s["scale_A"], s["scale_b"]
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    kind = st.kind
    if kind == "served":
        done, _ = serve.closed_loop(st.server, lambda i: st.scenes[i], len(st.scenes),
                                    len(st.scenes), keep_x=True)
        return [r["x"] for r in sorted(done, key=lambda r: r["tag"])]
    if kind == "batch":
        for solver, scene in zip(st.solvers, st.scenes):
            systems.assemble(solver, scene)
        st.batch.solve(st.solvers, max_iters=500, rel_tol=1e-12)
        return [s.x for s in st.solvers]
    if kind == "redistance":
        st.ls.phi.copy_(st.phi)
        st.ls.redistance()
        return st.ls.phi
    if kind == "extrapolate":
        for u, v in zip(st.velocity, st.given):
            u.copy_(v)
        projection.extrap_velocity(st.velocity, st.cell_type, iterations=10)
        return st.velocity
    if kind == "pressure":
        st.solver.reinitialize(st.scene["cell_type"], st.strategy)
        st.solver.solve(500, rel_tol=1e-12)
        return st.solver.x
    s = st.scene
    for u, v in zip(st.velocity, st.given):
        u.copy_(v)
    if kind == "volume":
        cells.apply_markers(st.cell_type, s["phi"])
        # the controller as the first substep left it
        st.strategy.step, st.strategy.vol_0, st.strategy.y = 1, st.target, 0.0
        st.solver.reinitialize(st.cell_type, st.strategy)
        st.solver.solve(500, rel_tol=1e-12)
        projection.apply_pressure(st.velocity, st.cell_type, st.solver.x, DT, RHO, s["dx"],
                                  s["p0"], ghost_fluid_method=True, phi=s["phi"],
                                  c_max=s["c_max"])
        return {"p": st.solver.x, "u": st.velocity}
    if kind == "surface":
        st.tension.solve_surface_tension()
        return st.velocity
    st.solver.full_reinitialize(st.potential)
    st.solver.solve(500, rel_tol=1e-18)
    psi = st.solver.x.clone()
    st.solver.reinitialize(s["cell_type"], st.strategy)
    st.solver.solve(500, rel_tol=1e-12)
    projection.apply_magnetic_force(st.velocity, st.cell_type, st.solver.x, st.H, DT, RHO,
                                    s["dx"], s["p0"], MU0, MAG_K)
    return {"psi": psi, "p": st.solver.x, "u": st.velocity}


def work(case):
    """Each input read once, each output written once; the solves' operations
    as one pass of a 7-point stencil."""
    boxes = _box_list(case) if case["kind"] in ("served", "batch") else [_res(case)]
    nbytes = flops = 0
    for res in boxes:
        n, d = math.prod(res), len(res)
        faces = sum(n // m * (m + 1) for m in res)
        per = {"redistance": 8 * n, "extrapolate": n + 8 * faces, "volume": 10 * n + 8 * faces,
               "surface": 4 * n + 8 * faces, "ferro": 21 * n + 12 * faces}
        nbytes += per.get(case["kind"], 12 * n + 4 * faces)  # cell types, phi, velocity; x
        flops += n * (2 * d + 1) * 2
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _shift(f, a, s, fill=0.0):
    """f at the neighbour s cells up axis a (fill outside)."""
    out = torch.full_like(f, fill)
    n = f.shape[a]
    if s > 0:
        out.narrow(a, 0, n - s).copy_(f.narrow(a, s, n - s))
    else:
        out.narrow(a, -s, n + s).copy_(f.narrow(a, 0, n + s))
    return out


def _sample(f, res, off):
    """f interpolated at every cell index plus off (clamped to the field)."""
    for a, n in enumerate(f.shape):
        pos = torch.arange(res[a], dtype=torch.float64, device=f.device) + off[a]
        i = pos.trunc().long().clamp(0, n - 1)
        w = (pos - i).clamp(0.0, 1.0).reshape([-1 if b == a else 1 for b in range(f.dim())])
        f = f.index_select(a, i) * (1 - w) + f.index_select(a, (i + 1).clamp(max=n - 1)) * w
    return f


def _cg(diag, upper, b, tol=1e-13, most=20000):
    """Jacobi-preconditioned conjugate gradients; rows with diag 0 are left out."""
    dim = b.dim()
    inv = torch.where(diag != 0, 1.0 / torch.where(diag != 0, diag, torch.ones_like(diag)), 0.0)

    def apply(v):
        out = diag * v
        for a in range(dim):
            n = v.shape[a]
            c = upper[a].narrow(a, 0, n - 1)
            out.narrow(a, 0, n - 1).addcmul_(c, v.narrow(a, 1, n - 1))
            out.narrow(a, 1, n - 1).addcmul_(c, v.narrow(a, 0, n - 1))
        return out

    x, r = torch.zeros_like(b), b.clone()
    z = inv * r
    p = z.clone()
    rz = (r * z).sum()
    stop = tol * float(b.norm())
    for i in range(most):
        q = apply(p)
        alpha = rz / (p * q).sum()
        x.add_(alpha * p)
        r.sub_(alpha * q)
        if i % 25 == 24 and float(r.norm()) <= stop:
            break
        z = inv * r
        new = (r * z).sum()
        p = z.add_(p * (new / rz))
        rz = new
    return x


def _pressure_exact(s, c=None, h2=None):
    """The pressure: cells coupled to fluid neighbours, air faces held at p0
    (ghost-fluid weighted; plus the magnetic pressure where h2 gives it)."""
    dim, ct, phi = s["dim"], s["cell_type"], s["phi"].double()
    sA, sb, p0 = s["scale_A"], s["scale_b"], s["p0"]
    fluid = ct == FLUID
    diag = torch.zeros_like(phi)
    div, rhs = torch.zeros_like(phi), torch.zeros_like(phi)
    upper = []
    for k in range(dim):
        u = s["velocity"][k].double()
        n = phi.shape[k]
        div += u.narrow(k, 0, n) - u.narrow(k, 1, n)
        for sgn in (-1, 1):
            nb = _shift(ct, k, sgn, SOLID)
            w = torch.ones_like(phi)
            if s["gfm"]:
                w = ((phi - _shift(phi, k, sgn)) / phi).clamp(max=s["c_max"])
                w = torch.where(phi == 0, torch.full_like(w, s["c_max"]), w)
            air = (nb == AIR) & fluid
            diag += sA * (nb == FLUID) + torch.where(air, sA * w, 0.0)
            jump = sA * w * p0 if h2 is None else sA * (p0 + 0.5 * MAG_K * MU0 * h2(k, sgn))
            rhs += torch.where(air, jump, 0.0)
            wall = u.narrow(k, 0, n) if sgn < 0 else u.narrow(k, 1, n)
            rhs += torch.where(nb == SOLID, sgn * sb * wall, 0.0)
        upper.append(torch.where(fluid & (_shift(ct, k, 1, SOLID) == FLUID), -sA, 0.0).double())
    b = div * sb + rhs + (c or 0.0)
    return _cg(torch.where(fluid, diag, 0.0), upper, torch.where(fluid, b, 0.0))


def _psi_exact(s, chi, H):
    dim, res, chi = s["dim"], s["res"], chi.double()
    diag, b = torch.zeros_like(chi), torch.zeros_like(chi)
    upper = []
    for k in range(dim):
        n = res[k]
        up = torch.zeros_like(chi)
        mean = 0.5 * (chi.narrow(k, 0, n - 1) + chi.narrow(k, 1, n - 1))
        up.narrow(k, 0, n - 1).copy_((1 + mean) / s["dx"])
        diag -= up + _shift(up, k, -1)
        upper.append(up)
        flux = _sample(chi, res, [0.0 if a == k else 0.5 for a in range(dim)]) * \
            H[k].double().narrow(k, 0, n)
        flux.select(k, 0).zero_()
        b += _shift(flux, k, 1) - flux
    at = (0,) * dim
    b[at] = 0.0
    diag[at] = 1.0 / s["dx"]
    for up in upper:
        up[at] = 0.0
    # the reference row alone fixes psi(0) = 0, so its couplings may go: the
    # neighbours' rows keep theirs on the diagonal, which makes the rest definite
    return _cg(diag, upper, b)


def _delta(phi, dx):
    eps = 5 * dx
    return torch.where(phi.abs() < eps, (1 + torch.cos(math.pi * phi / eps)) / (2 * eps), 0.0)


def _surface_exact(s, d, u):
    """The implicit capillary step of component d."""
    dim, res, dx = s["dim"], s["res"], s["dx"]
    phi, u = s["phi"].double(), u.double()
    half = [0.0 if a == d else 0.5 for a in range(dim)]

    def at(f, *moves, base=None):
        off = list(base or [0.0] * dim)
        for a, h in moves:
            off[a] += h
        return _sample(f, res, off)

    grad = [(at(phi, (k, 0.5), base=half) - at(phi, (k, -0.5), base=half)) / dx
            for k in range(dim)]
    norm = sum(g * g for g in grad).sqrt()
    n = [torch.where(norm > 0, g / torch.where(norm > 0, norm, torch.ones_like(norm)), 0.0)
         for g in grad]
    kappa = sum((at(n[k], (k, 0.5)) - at(n[k], (k, -0.5))) / dx for k in range(dim))
    du = sum((at(u, (k, 0.5)) - at(u, (k, -0.5))) / dx * n[k] for k in range(dim))
    d2 = 0.0
    for i in range(dim):
        for j in range(dim):
            m = (at(u, (i, 0.5), (j, 0.5)) + at(u, (i, -0.5), (j, -0.5)) -
                 at(u, (i, 0.5), (j, -0.5)) - at(u, (i, -0.5), (j, 0.5))) / dx ** 2
            d2 = d2 + n[i] * m * n[j]
    b = u.narrow(d, 0, res[d]) / DT - SIGMA * _delta(at(phi, base=half), dx) * \
        (kappa * n[d] + DT * (d2 + kappa * du))
    diag = torch.full_like(b, 1.0 / DT)
    upper = []
    for k in range(dim):
        w = SIGMA * DT / dx ** 2 * _delta(at(phi, (k, 0.5), base=half), dx)
        w.select(k, res[k] - 1).zero_()
        diag += w + _shift(w, k, -1)
        upper.append(-w)
    return _cg(diag, upper, b)


def _volume(phi, dx):
    """The fluid's volume in cells: the smoothed step at every cell's corners."""
    eps, tot = 5 * dx, 0.0
    corners = 1 << phi.dim()
    for o in range(corners):
        v = -_sample(phi, phi.shape, [(o >> a & 1) - 0.5 for a in range(phi.dim())])
        mid = 0.5 + v / (2 * eps) + torch.sin(math.pi * v / eps) / (2 * math.pi)
        step = torch.where(v <= -eps, 0.0, torch.where(v >= eps, 1.0, mid))
        tot += float(step.sum()) / corners
    return tot


def _project_exact(s, ct, p, jump_up, jump_down):
    """The velocity after the pressure gradient: 0 at walls, the air side of a
    fluid-air face from jump_up (fluid below) or jump_down (fluid above)."""
    scale = DT / (RHO * s["dx"])
    out = []
    for k in range(s["dim"]):
        u = s["velocity"][k].double().clone()
        n = ct.shape[k]
        below, pl = _shift(ct, k, -1, SOLID), _shift(p, k, -1)
        v = u.narrow(k, 0, n)
        new = torch.where((ct == FLUID) & (below == FLUID), v - scale * (p - pl), v)
        new = torch.where((ct == AIR) & (below == FLUID), v - scale * jump_up(k, pl), new)
        new = torch.where((ct == FLUID) & (below == AIR), v - scale * jump_down(k, p), new)
        wall = ((ct == FLUID) & (below == SOLID)) | ((ct == SOLID) & (below == FLUID))
        v.copy_(torch.where(wall, 0.0, new))
        out.append(u)
    return out


def _redistance_exact(phi, dx, repeats=2):
    """Fast sweeping: cells at the zero crossing fixed, then one sweep up and
    one down each axis, the last axis first; a sweep reads the lines beside it
    as they were before it."""
    dim = phi.dim()
    sgn = torch.sign(phi)
    est = torch.full_like(phi, 1e20)
    fixed = torch.zeros_like(phi, dtype=torch.bool)
    for k in range(dim):
        for s in (-1, 1):
            pj = _shift(phi, k, s)
            cross = (sgn != torch.sign(pj)) & (_shift(torch.ones_like(phi), k, s) > 0)
            e = sgn * (phi / (phi - pj)) * dx
            est = torch.where(cross & (e.abs() < est.abs()), e, est)
            fixed |= cross
    tmp = torch.where(fixed, est, torch.full_like(est, 1e20))
    for _ in range(repeats):
        for ax in reversed(range(dim)):
            line = [a for a in range(dim) if a != ax]
            order = [ax] + line
            sg = sgn.permute(order).contiguous()
            fx = fixed.permute(order).contiguous()
            for up in (True, False):
                live = tmp.permute(order).contiguous()
                across = [torch.minimum(_shift(live.abs(), a + 1, -1, math.inf),
                                        _shift(live.abs(), a + 1, 1, math.inf))
                          for a in range(len(line))]
                n = live.shape[0]
                for i in (range(n) if up else reversed(range(n))):
                    lo = live[i - 1].abs() if i > 0 else None
                    hi = live[i + 1].abs() if i + 1 < n else None
                    along = hi if lo is None else lo if hi is None else torch.minimum(lo, hi)
                    nb = torch.sort(torch.stack([along] + [f[i] for f in across]), dim=0).values
                    d = nb[0] + dx
                    two = 0.5 * (nb[0] + nb[1] + (2 * dx * dx - (nb[1] - nb[0]) ** 2)
                                 .clamp(min=0.0).sqrt())
                    if dim == 3:
                        tot = nb[0] + nb[1] + nb[2]
                        q = nb[0] ** 2 + nb[1] ** 2 + nb[2] ** 2 - dx * dx
                        three = (tot + (tot * tot - 3 * q).clamp(min=0.0).sqrt()) / 3
                        two = torch.where(two > nb[2], three, two)
                    d = torch.where(d > nb[1], two, d)
                    better = (d < live[i].abs()) & ~fx[i]
                    live[i] = torch.where(better, d * sg[i], live[i])
                inverse = [order.index(a) for a in range(dim)]
                tmp = live.permute(inverse).contiguous()
    return tmp


def _extrapolate_exact(u, k, ct, iterations):
    u = u.double().clone()
    n = ct.shape[k]
    fluid = torch.zeros_like(u)
    fluid.narrow(k, 0, n).add_((ct == FLUID).double())
    fluid.narrow(k, 1, n).add_((ct == FLUID).double())
    valid = (fluid > 0).double()

    def block(f):
        for a in range(f.dim()):
            f = f + _shift(f, a, 1) + _shift(f, a, -1)
        return f

    for _ in range(iterations):
        tot, cnt = block(u * valid), block(valid)
        grow = (valid == 0) & (cnt > 0)
        u = torch.where(grow, tot / cnt.clamp(min=1.0), u)
        valid = torch.where(grow, torch.ones_like(valid), valid)
    return u


def _scene_exact(s):
    if s["kind"] == "psi":
        return _psi_exact(s, s["chi"], s["H_ext"])
    if s["kind"] == "surface":
        return _surface_exact(s, s["d"], s["velocity"][s["d"]])
    return _pressure_exact(s, s.get("c"))


def exact(case, seed):
    kind = case["kind"]
    if kind in ("served", "batch"):
        return [_scene_exact(s) for s in _scenes(case, seed)]
    res = _res(case)
    dim = len(res)
    if kind == "redistance":
        dx, phi = _advected(res, seed)
        return _redistance_exact(phi.double(), dx)
    if kind == "extrapolate":
        _, phi = _pool(res, seed, 2)
        ct = _cell_types(phi, torch.int8)
        return [_extrapolate_exact(u, k, ct, 10)
                for k, u in enumerate(_faces(res, _generator(seed)))]
    if kind == "pressure":
        return _pressure_exact(_scene("pressure", res, seed, case["spheres"], case["gfm"],
                                      case["L"]))
    s = _scene("pressure", res, seed, 2, True, case["L"])
    if kind == "surface":
        out = []
        for k, u in enumerate(s["velocity"]):
            v = u.double().clone()
            v.narrow(k, 0, res[k]).copy_(_surface_exact(s, k, u))
            out.append(v)
        return out
    phi, ct = s["phi"].double(), s["cell_type"]
    if kind == "volume":
        s["c_max"] = 1e3
        target = 1.01 * float((s["phi"] <= 0).sum().item())
        x = (_volume(phi, s["dx"]) - target) / target
        k_p = 2.3 / (25 * DT)
        c = (-k_p * x - (k_p / 4) ** 2 * x * DT) / (x + 1)
        p = _pressure_exact(s, c)

        def weight(k, here, there):
            w = ((here - there) / here).clamp(max=s["c_max"])
            return torch.where(here == 0, torch.full_like(w, s["c_max"]), w)

        def jump_up(k, pl):
            return (s["p0"] - pl) * weight(k, _shift(phi, k, -1), phi)

        def jump_down(k, ph):
            return (ph - s["p0"]) * weight(k, phi, _shift(phi, k, -1))

        return {"p": p, "u": _project_exact(s, ct, p, jump_up, jump_down)}
    # ferro
    H = [h.double() for h in _magnet(res, s["dx"], seed)]
    chi = torch.where(s["phi"] <= 0, 2.0, 0.0)

    def h2(off):
        return sum(_sample(H[a], res, [o - (0.0 if a == b else 0.5) for b, o in enumerate(off)])
                   ** 2 for a in range(dim))

    p = _pressure_exact(s, None, lambda k, sgn: h2([0.5 + (sgn if a == k else 0)
                                                    for a in range(dim)]))

    def air(k, below):
        off = [0.5 - (1 if below and a == k else 0) for a in range(dim)]
        return s["p0"] + 0.5 * MAG_K * MU0 * h2(off)

    u = _project_exact(s, ct, p, lambda k, pl: air(k, False) - pl,
                       lambda k, ph: ph - air(k, True))
    return {"psi": _psi_exact(s, chi, H), "p": p, "u": u}
