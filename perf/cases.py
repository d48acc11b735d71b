"""Workloads of the MI355X cell residual, as a user's program runs them.

Each case is one call (or one fixed sequence of calls) through the public
entry points of ibis_amd:

  residual   FiniteVolume.compute_dudt
  rk         RungeKutta.take_step, one ssp-rk3 step, dt returned to the host
  batch      Batch.rk_steps, many independent instances stepped together
  vjp        FiniteVolume.compute_dudt_vjp, the discrete adjoint
  autograd   autograd.residual and autograd.wall_force, forward and backward
  jvp        FiniteVolume.compute_dudt_jvp, the tangent residual
  matvec     SteadyStateLinearisation.matrix_vector_product
  jfnk       Jfnk.initialise and one Jfnk.step (GMRES or FGMRES)

on the grids of ibis_amd.gridgen: the 2D wedge and ramp, the viscous flat
plate, and the jittered hex box whose cells are stored in random order.

``exact`` evaluates the same quantities with plain torch operations in 64
bits on the cells in the order of the grid file, with the derivatives by
torch's automatic differentiation; only the permutation of the cells to the
grid's numbering (integers) is taken from the grid.
"""
import functools
import math

import numpy as np
import torch

from ibis_amd import autograd, gridgen
from ibis_amd import cases as workloads
from ibis_amd import config as C
from ibis_amd.batch import Batch
from ibis_amd.finite_volume import FiniteVolume, GridBlock, RungeKutta
from ibis_amd.steady import Jfnk, SteadyStateLinearisation

F64 = torch.float64
DEV = "cuda"
RHO, P, T, E, VX, VY, VZ = range(7)


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def _case(what, mesh, nx, ny=0, **kw):
    c = {"what": what, "mesh": mesh, "nx": nx, "ny": ny, "mach": 3.0, "angle": 15.0,
         "flux": "hanel" if mesh == "hex" else "ausmdv",
         "limiter": "venkatakrishnan" if mesh == "hex" else "barth_jespersen",
         "thermo": "rho_u", "precision": "fp64"}
    c.update(kw)
    return c


def listed():
    return [
        # the smallest call: a coarse grid while a job is set up; what counts
        # is the latency of the launches and of the chains inside them
        dict(_case("residual", "wedge", 48, 24), name="residual_wedge_48x24"),
        # the explicit solver of a 2D transient job, 18k cells, one step with
        # its dt back on the host
        dict(_case("rk", "wedge", 192, 96), name="rk_wedge_192x96"),
        # a parameter study: 16 small wedges and ramps of uneven size, 10 steps
        # a call on the device
        dict(_case("batch", "wedge", 16, cells_min=1000, cells_max=20000, steps=10),
             name="batch_16"),
        # the viscous residual of a boundary-layer grid, 0.5M cells
        dict(_case("residual", "plate", 1024, 512, mach=2.0), name="residual_plate_1024x512"),
        # one adjoint solve's operator on that grid: dU/dt cotangent and wall force
        dict(_case("vjp", "plate", 1024, 512, mach=2.0, mode="active"),
             name="vjp_plate_1024x512"),
        # a gradient of a loss through torch.autograd on an odd-sized ramp
        dict(_case("autograd", "ramp", 301, 151, mach=2.5, angle=9.0, flux="hanel",
                   limiter="venkatakrishnan", thermo="rho_p", mode="active"),
             name="autograd_ramp_301x151"),
        # the 3D residual at scale, 2.1M cells, and in the reduced-precision
        # mode on an odd-sized box
        dict(_case("residual", "hex", 128), name="residual_hex_128"),
        dict(_case("residual", "hex", 75, precision="fp32_recon"), name="residual_hex_75_fp32"),
        # sensitivities by forward differentiation on a 3D box
        dict(_case("jvp", "hex", 48), name="jvp_hex_48"),
        # the operator that the steady solver's Krylov method applies, viscous
        dict(_case("matvec", "plate", 512, 256, mach=2.0), name="matvec_plate_512x256"),
        # a pseudo-transient step of the steady solver: GMRES on the wedge,
        # preconditioned FGMRES on a small plate
        dict(_case("jfnk", "wedge", 192, 96, solver="gmres", iters=30, tol=1e-3, cfl=10.0),
             name="jfnk_gmres_wedge_192x96"),
        dict(_case("jfnk", "plate", 96, 48, mach=2.0, solver="fgmres", iters=8, tol=1e-3,
                   cfl=10.0, inner_iters=8, inner_tol=1e-1), name="jfnk_fgmres_plate_96x48"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["residual", "residual", "residual", "rk", "rk", "batch", "vjp", "autograd",
                       "jvp", "matvec", "matvec", "jfnk"])
    flux = rng.choice(["ausmdv", "hanel", "rusanov"])
    limiter = rng.choice(["barth_jespersen", "venkatakrishnan"])
    thermo = rng.choice(["rho_u", "rho_p", "rho_T", "p_T"])
    opt = {"flux": flux, "limiter": limiter, "thermo": thermo}
    if what == "batch":
        lo = _log_int(rng, 300, 4000)
        return _case("batch", "wedge", rng.randint(3, 24), cells_min=lo,
                     cells_max=lo * rng.randint(2, 6), steps=rng.randint(2, 12), **opt)
    meshes = {"residual": ["wedge", "ramp", "plate", "hex"], "rk": ["wedge", "ramp", "plate"],
              "vjp": ["plate", "hex", "wedge"], "autograd": ["ramp", "wedge", "plate"],
              "jvp": ["hex", "wedge", "plate"], "matvec": ["wedge", "plate", "hex"],
              "jfnk": ["wedge", "plate"]}
    mesh = rng.choice(meshes[what])
    if mesh == "hex":
        kw = dict(opt)
        if what == "residual":
            kw["precision"] = rng.choice(["fp64", "fp64", "fp32_flux", "fp32_recon"])
        if what == "vjp":
            kw["mode"] = rng.choice(["active", "frozen"])
        return _case(what, "hex", _log_int(rng, 8, {"residual": 96, "vjp": 56}.get(what, 48)), **kw)
    top = {"residual": 500_000, "rk": 200_000, "vjp": 250_000, "autograd": 120_000,
           "jvp": 130_000, "matvec": 130_000, "jfnk": 18_000}[what]
    cells = _log_int(rng, 700 if what != "jfnk" else 400, top)
    ny = max(7, int(round(math.sqrt(cells / 2.0))))
    nx = max(9, cells // ny)
    kw = dict(opt, mach=round(rng.uniform(1.8, 3.5), 3), angle=round(rng.uniform(5.0, 15.0), 3))
    if mesh == "plate":
        kw["mach"] = 2.0
    if what in ("vjp", "autograd"):
        kw["mode"] = rng.choice(["active", "frozen"])
    if what == "jfnk":
        kw.update(solver=rng.choice(["gmres", "fgmres"]), iters=rng.randint(4, 12), tol=1e-3,
                  cfl=round(rng.uniform(2.0, 10.0), 2), inner_iters=rng.randint(2, 8),
                  inner_tol=1e-1)
    return _case(what, mesh, nx, ny, **kw)


# ---------------------------------------------------------------------------
# grids, configurations and states
# ---------------------------------------------------------------------------
def _freestream(c):
    return (workloads.plate_freestream(c["mach"]) if c["mesh"] == "plate"
            else workloads.freestream(c["mach"]))


def _grid_and_config(c):
    fs = _freestream(c)
    if c["mesh"] == "hex":
        g, cfg = workloads.hex_case(c["nx"], flux=c["flux"], limiter=c["limiter"])
    elif c["mesh"] == "plate":
        g = gridgen.flat_plate(c["nx"], c["ny"])
        cfg = workloads.plate_config(fs, flux=c["flux"])
    else:
        make = gridgen.wedge if c["mesh"] == "wedge" else gridgen.ramp
        g = make(c["nx"], c["ny"], angle_deg=c["angle"])
        cfg = workloads.wedge_config(fs, flux=c["flux"])
    cfg.limiter, cfg.thermo_interpolator = c["limiter"], c["thermo"]
    return g, cfg


@functools.lru_cache(maxsize=3)
def _operator(key):
    """Grid, operator and cell permutation of a case: what a program builds
    once and keeps while it evaluates many states."""
    c = dict(key)
    g, cfg = _grid_and_config(c)
    gb = GridBlock(g, cfg, reorder=True)
    fv = FiniteVolume(gb, cfg)
    if c["precision"] != "fp64":
        fv.set_precision(c["precision"])
    return g, cfg, gb, fv, torch.from_numpy(gb.cell_new_of_old).to(DEV)


def _key(c):
    return tuple((k, c[k]) for k in ("mesh", "nx", "ny", "mach", "angle", "flux", "limiter",
                                     "thermo", "precision"))


def _centres(g):
    nv = 8 if g.dim == 3 else 4
    xyz = torch.from_numpy(g.xyz).to(DEV)
    return xyz[torch.from_numpy(g.cvtx[:, :nv].copy()).to(DEV)].mean(dim=1)


def _waves(rng, x, count):
    """Sums of three sinusoids in [-1, 1] with wave numbers and phases from rng."""
    L = float((x.max(dim=0).values - x.min(dim=0).values).max())
    out = []
    for _ in range(count):
        s = 0.0
        for m in range(3):
            k = rng.uniform(0.6, 1.4, 3) * (1.0 + m)
            s = s + torch.sin(2 * math.pi / L * (k[0] * x[:, 0] + k[1] * x[:, 1] + k[2] * x[:, 2])
                              + 2 * math.pi * rng.random()) / 3.0
        out.append(s)
    return out


def _state(c, g, n_ghost, seed):
    """7 x N_total primitive state in the grid file's cell order: a smooth
    seeded field around the free stream (the hex box: Mach 0.3 to 3 in every
    direction); ghost cells start at the free stream."""
    fs, gas = _freestream(c), C.IdealGas()
    rng = np.random.default_rng([seed, 17])
    x = _centres(g)
    n = x.shape[0]
    w = _waves(rng, x, 6)
    s = torch.empty((7, n + n_ghost), dtype=F64, device=DEV)
    s[:, n:] = torch.tensor([fs.rho, fs.p, fs.T, fs.energy, fs.vx, fs.vy, fs.vz], dtype=F64,
                            device=DEV)[:, None]
    if c["mesh"] == "hex":
        rho, p = 1.2 * (1 + 0.2 * w[0]), 1e5 * (1 + 0.2 * w[1])
        temp = p / (rho * gas.R)
        speed = (1.65 + 1.35 * w[2]) * torch.sqrt(gas.gamma * gas.R * temp)
        norm = torch.sqrt(w[3] ** 2 + w[4] ** 2 + w[5] ** 2) + 1e-3
        vel = [speed * w[3 + k] / norm for k in range(3)]
    else:
        u = math.hypot(fs.vx, fs.vy)
        rho, temp = fs.rho * (1 + 0.05 * w[0]), fs.T * (1 + 0.05 * w[1])
        p = rho * gas.R * temp
        vel = [fs.vx + 0.05 * u * w[2], fs.vy + 0.05 * u * w[3], torch.zeros_like(p)]
    for row, v in zip(range(7), (rho, p, temp, gas.Cv * temp, *vel)):
        s[row, :n] = v
    return s


def _scale(c):
    """Sizes of the state's rows: the scales of tangents and cotangents."""
    fs = _freestream(c)
    u = math.hypot(fs.vx, fs.vy)
    return torch.tensor([fs.rho, fs.p, fs.T, fs.energy, u, u, u if c["mesh"] == "hex" else 0.0],
                        dtype=F64, device=DEV)[:, None]


def _vector(c, g, n_ghost, seed):
    """A smooth perturbation of the valid cells' state (7 x N_total) and a
    cotangent of dU/dt ((dim+2) x N_total), both in the grid file's order."""
    rng = np.random.default_rng([seed, 29])
    x = _centres(g)
    n = x.shape[0]
    w = torch.stack(_waves(rng, x, 7 + g.dim + 2))
    dot = torch.zeros((7, n + n_ghost), dtype=F64, device=DEV)
    dot[:, :n] = 1e-2 * _scale(c) * w[:7]
    bar = torch.zeros((g.dim + 2, n + n_ghost), dtype=F64, device=DEV)
    bar[:, :n] = w[7:]
    return dot, bar


def _instances(c):
    out = []
    for k, spec in enumerate(workloads.batch_instances(n=c["nx"], seed=7, n_min=c["cells_min"],
                                                       n_max=c["cells_max"])):
        out.append(dict(c, mesh=spec["kind"], nx=spec["nx"], ny=spec["ny"],
                        angle=round(spec["angle"], 3), mach=round(spec["mach"], 3)))
    return out


def _cons(s, dim):
    rho, v = s[RHO], s[VX:VX + 3]
    rows = [rho] + [rho * v[k] for k in range(dim)]
    ke = 0.5 * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2])
    return torch.stack(rows + [rho * (ke + s[E])])


def _solver_json(c):
    if c["solver"] == "gmres":
        ls = {"type": "gmres", "max_iters": c["iters"], "tol": c["tol"]}
    else:
        ls = {"type": "fgmres", "max_iters": c["iters"], "tolerance": c["tol"],
              "max_preconditioner_iters": c["inner_iters"],
              "preconditioner_tolerance": c["inner_tol"]}
    return {"max_steps": 1, "tolerance": 1e-10, "linear_solver": ls,
            "cfl": {"type": "constant", "value": c["cfl"]}}


def _ordered(a, new_of_old):
    out = torch.empty_like(a)
    out[:, new_of_old] = a
    return out


def _cell_major(a, n):
    """(rows, N_total) -> the Krylov vectors' order, cell * rows + row."""
    return a[:, :n].T.contiguous().reshape(-1)


# ---------------------------------------------------------------------------
# what a program has in hand, and one pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    c = case
    if c["what"] == "batch":
        inst = _instances(c)
        grids = [_grid_and_config(i) for i in inst]
        b = Batch(grids, reorder=True)
        prim = torch.zeros((7, b.Nt), dtype=F64, device=DEV)
        for k, i in enumerate(inst):
            cols = torch.from_numpy(b.columns(k)).to(DEV)
            order = torch.from_numpy(b.blocks[k].cell_new_of_old).to(DEV)
            prim[:, cols] = _ordered(_state(i, grids[k][0], b.blocks[k].G, seed + 100 * k), order)
        cons = _cons(prim, 2).contiguous()
        b.rk_init(cons, prim, cfl=0.5)
        return {"c": c, "batch": b, "cons": cons, "prim": prim}
    g, cfg, gb, fv, order = _operator(_key(c))
    st = {"c": c, "gb": gb, "fv": fv}
    ref = _state(c, g, gb.G, seed)
    st["prim"] = _ordered(ref, order)
    nc = gb.dim + 2
    what = c["what"]
    if what in ("residual", "autograd", "jvp"):
        st["dudt"] = torch.zeros((nc, gb.Nt), dtype=F64, device=DEV)
    if what in ("rk", "matvec", "jfnk"):
        st["cons"] = _cons(st["prim"], gb.dim).contiguous()
    if what in ("vjp", "autograd", "jvp", "matvec"):
        dot, bar = _vector(c, g, gb.G, seed)
        st["dot"], st["bar"] = _ordered(dot, order), _ordered(bar, order)
    if what == "rk":
        st["rk"] = RungeKutta(fv, method="ssp-rk3", cfl=0.5)
    elif what == "vjp":
        st["prim_bar"] = torch.zeros_like(st["prim"])
        st["tags"] = fv.tag_mask(_force_tag(c))
    elif what == "autograd":
        st["tags"] = fv.tag_mask(_force_tag(c))
    elif what == "jvp":
        st["dudt_dot"] = torch.zeros_like(st["dudt"])
    elif what == "matvec":
        st["op"] = SteadyStateLinearisation(fv, st["cons"])
        st["op"].set_pseudo_time_step(_DT_STAR)
        dcons = torch.func.jvp(lambda s: _cons(s, gb.dim), (st["prim"],), (st["dot"],))[1]
        st["vec"] = _cell_major(dcons, gb.N)
        st["result"] = torch.zeros_like(st["vec"])
    elif what == "jfnk":
        st["cons0"], st["prim0"] = st["cons"].clone(), st["prim"].clone()
        st["solver"] = Jfnk(fv, _solver_json(c))
    return st


_DT_STAR = 1e-5  # pseudo time step of the matvec cases, in seconds
_FORCE_DIR = (1.0, 0.25, 0.0)


def _force_tag(c):
    return "bottom" if c["mesh"] == "hex" else "wall"


def run(state):
    st, c = state, state["c"]
    what = c["what"]
    if what == "batch":
        st["batch"].rk_steps(c["steps"])
        return {"cons": st["cons"], "prim": st["prim"]}
    fv, gb, prim = st["fv"], st["gb"], st["prim"]
    if what == "residual":
        fv.compute_dudt(prim, gb, st["dudt"])
        return {"dudt": st["dudt"], "prim": prim}
    if what == "rk":
        dt = st["rk"].take_step(st["cons"], prim)
        return {"cons": st["cons"], "prim": prim, "dt": dt}
    if what == "vjp":
        fv.compute_dudt_vjp(prim, st["prim_bar"], dudt_bar=st["bar"], force_tags=st["tags"],
                            force_dir=_FORCE_DIR, limiter=c["mode"])
        return {"prim_bar": st["prim_bar"], "prim": prim}
    if what == "autograd":
        x = prim.detach().requires_grad_(True)
        r = autograd.residual(x, fv, c["mode"])
        j = autograd.wall_force(x, fv, st["tags"], _FORCE_DIR, c["mode"])
        (grad,) = torch.autograd.grad((r * st["bar"]).sum() + j, x)
        return {"dudt": r.detach(), "force": j.detach(), "grad": grad}
    if what == "jvp":
        fv.compute_dudt_jvp(prim, st["dot"], st["dudt"], st["dudt_dot"])
        return {"dudt": st["dudt"], "dudt_dot": st["dudt_dot"], "prim": prim, "dot": st["dot"]}
    if what == "matvec":
        st["op"].matrix_vector_product(st["vec"], st["result"])
        return {"result": st["result"]}
    # a steady solve starts from its initial state
    st["cons"].copy_(st["cons0"])
    prim.copy_(st["prim0"])
    st["solver"].initialise(st["cons"], prim)
    res = st["solver"].step(st["cons"], prim, 0)
    return {"cons": st["cons"], "prim": prim, "iters": res.n_iters,
            "norms": [float(v) for v in st["solver"].residual_norms().values()]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _counts(c):
    """dim, cells, all cells, faces, faces per cell, LSQ factors."""
    if c["mesh"] == "hex":
        n = c["nx"]
        return 3, n ** 3, n ** 3 + 6 * n * n, 3 * n * n * (n + 1), 6, 6
    nx, ny = c["nx"], c["ny"]
    return 2, nx * ny, nx * ny + 2 * (nx + ny), nx * (ny + 1) + ny * (nx + 1), 4, 3


def _residual_work(c):
    """Bytes: the state and dU/dt, volumes, centroids, LSQ factors, face
    geometry and connectivity once each.  Operations: gradients, limiter and
    reconstruction per cell, flux (and viscous terms) per face."""
    dim, n, nt, f, nf, nl = _counts(c)
    nc = dim + 2
    geom = n * 8 * (dim + 1 + nl) + f * (16 * dim + 16) + n * (4 * nf + 4)
    flops = n * (nf * (5 * 30 + 20) + 60) + f * 150
    if c["mesh"] == "plate":
        flops += n * nf * 40 + f * 120
    return 8 * nc * nt, 8 * nc * n, geom, flops


def work(case):
    c, what = case, case["what"]
    if what == "batch":
        parts = [_residual_work(i) for i in _instances(c)]
        s, d, geom, fl = (sum(p[k] for p in parts) for k in range(4))
        return {"bytes": 4 * s + geom, "flops": 3 * c["steps"] * fl}
    s, d, geom, fl = _residual_work(c)
    if what == "rk":
        return {"bytes": 4 * s + geom, "flops": 3 * fl}
    if what == "residual":
        return {"bytes": s + d + geom, "flops": fl}
    if what == "vjp":
        return {"bytes": 2 * s + d + geom, "flops": 3 * fl}
    if what == "autograd":
        return {"bytes": 3 * s + 2 * d + geom, "flops": 4 * fl}
    if what == "jvp":
        return {"bytes": 2 * (s + d) + geom, "flops": 3 * fl}
    if what == "matvec":
        return {"bytes": s + 2 * d + geom, "flops": 3 * fl}
    # the operator's inputs once per Krylov vector and the basis once
    k = c["iters"] * (c["inner_iters"] if c["solver"] == "fgmres" else 1)
    return {"bytes": k * (s + 2 * d + geom), "flops": k * 3 * fl}


# ---------------------------------------------------------------------------
# the same quantities in plain torch, 64 bits
# ---------------------------------------------------------------------------
_QUAD_FACES = ((0, 1), (1, 2), (2, 3), (3, 0))
_HEX_FACES = ((0, 1, 2, 3), (0, 1, 5, 4), (4, 5, 6, 7), (2, 3, 7, 6), (0, 4, 7, 3), (1, 5, 6, 2))


def _cross(a, b):
    return torch.stack([a[:, 1] * b[:, 2] - a[:, 2] * b[:, 1],
                        a[:, 2] * b[:, 0] - a[:, 0] * b[:, 2],
                        a[:, 0] * b[:, 1] - a[:, 1] * b[:, 0]], dim=1)


def _norm(a):
    return torch.sqrt((a * a).sum(dim=1))


def _quad_area(p, q, r, s):
    return 0.5 * _norm(_cross(q - p, r - p)) + 0.5 * _norm(_cross(r - p, s - p))


class _Mesh:
    """Faces, cells and ghosts of a grid of quads or of hexes, numbered in
    the grid file's order; lists per cell are (cells, faces per cell)."""

    def __init__(self, g, cfg):
        dev = torch.device(DEV)
        self.dim = g.dim
        local = torch.tensor(_HEX_FACES if g.dim == 3 else _QUAD_FACES, device=dev)
        xyz = torch.from_numpy(g.xyz).to(dev)
        cv = torch.from_numpy(g.cvtx[:, :8 if g.dim == 3 else 4].copy()).to(dev)
        self.N = N = cv.shape[0]
        verts = cv[:, local]                                  # N, nf, vertices of a face
        nf, k = local.shape
        flat = verts.reshape(N * nf, k)
        big = int(xyz.shape[0]) + 1

        def keys(v):  # smallest and largest vertex: unique on these structured grids
            return v.min(dim=1).values * big + v.max(dim=1).values

        _, inv = torch.unique(keys(flat), return_inverse=True)
        F = int(inv.max()) + 1
        first = torch.full((F,), N * nf, dtype=torch.int64, device=dev)
        first.scatter_reduce_(0, inv, torch.arange(N * nf, device=dev), "amin")
        rank = torch.empty_like(first)
        rank[first.argsort()] = torch.arange(F, device=dev)
        self.cell_faces = rank[inv].reshape(N, nf)
        self.F = F
        fv = flat[first.sort().values]                        # vertices as the first cell lists them
        p = [xyz[fv[:, q]] for q in range(k)]
        self.xf = sum(p) / k
        t1 = p[1] - p[0]
        t1 = t1 / _norm(t1)[:, None]
        if g.dim == 3:
            d = p[2] - p[0]
            t2 = d - (t1 * d).sum(dim=1, keepdim=True) * t1
            t2 = t2 / _norm(t2)[:, None]
            self.area = _quad_area(*p)
        else:
            t2 = torch.tensor([0.0, 0.0, 1.0], dtype=F64, device=dev).expand_as(t1)
            self.area = _norm(p[1] - p[0])
        self.n, self.t1, self.t2 = _cross(t1, t2), t1, t2
        xc = xyz[cv].mean(dim=1)
        out = ((self.xf[self.cell_faces] - xc[:, None]) * self.n[self.cell_faces]).sum(dim=2) > 0
        self.sign = torch.where(out, 1.0, -1.0).to(F64)
        L = torch.full((F,), -1, dtype=torch.int64, device=dev)
        R = torch.full((F,), -1, dtype=torch.int64, device=dev)
        cells = torch.arange(N, device=dev)[:, None].expand(N, nf)
        L[self.cell_faces[out]] = cells[out]
        R[self.cell_faces[~out]] = cells[~out]
        # ghosts by sorted tag, in the order of the markers' elements
        sorted_keys, at = keys(fv).sort()
        self.tags, ghost = [], N
        for name in cfg.tags():
            bv = torch.from_numpy(g.markers[name][1][:, :k].copy()).to(dev)
            f = at[torch.searchsorted(sorted_keys, keys(bv))]
            ids = torch.arange(ghost, ghost + len(f), device=dev)
            ghost += len(f)
            left = L[f] < 0
            L[f[left]], R[f[~left]] = ids[left], ids[~left]
            self.tags.append((name, f, torch.where(left, R[f], L[f]), ids))
        self.L, self.R, self.Nt = L, R, ghost
        self.xc = torch.empty((ghost, 3), dtype=F64, device=dev)
        self.xc[:N] = xc
        for _, f, valid, ids in self.tags:
            self.xc[ids] = 2.0 * self.xf[f] - xc[valid]
        cf = self.cell_faces
        self.nbr = torch.where(L[cf] == cells, R[cf], L[cf])
        if g.dim == 3:  # (1/3) sum of x_f . n A, about the origin
            self.vol = (self.sign * (self.xf * self.n).sum(dim=1)[cf] * self.area[cf]).sum(dim=1) / 3
        else:
            self.vol = _quad_area(*[xyz[cv[:, q]] for q in range(4)])
        # least-squares weights of each neighbour (QR factors; the 3D beta
        # is the reference's own expression, gradient.h:89)
        d = self.xc[self.nbr] - self.xc[:N, None]
        sxx, sxy, sxz = [(d[..., 0] * d[..., q]).sum(dim=1) for q in range(3)]
        syy, syz = [(d[..., 1] * d[..., q]).sum(dim=1) for q in (1, 2)]
        szz = (d[..., 2] * d[..., 2]).sum(dim=1)
        r11 = torch.sqrt(sxx)
        r12 = sxy / r11
        r22 = torch.sqrt(syy - r12 * r12)
        a1 = d[..., 0] / (r11 * r11)[:, None]
        a2 = (d[..., 1] - (r12 / r11)[:, None] * d[..., 0]) / (r22 * r22)[:, None]
        w = torch.zeros((N, nf, 3), dtype=F64, device=dev)
        w[..., 0], w[..., 1] = a1 - (r12 / r11)[:, None] * a2, a2
        if g.dim == 3:
            r13 = sxz / r11
            r23 = (syz - r12 / r11 * sxz) / r22
            r33 = torch.sqrt(szz - r13 * r13 - r23 * r23)
            beta = ((r12 * r23 - r13 * r23) / (r11 * r22))[:, None]
            a3 = (d[..., 2] - (r23 / r22)[:, None] * d[..., 1] + beta * d[..., 0]) / (r33 * r33)[:, None]
            w[..., 0] = w[..., 0] + beta * a3
            w[..., 1] = w[..., 1] - (r23 / r22)[:, None] * a3
            w[..., 2] = a3
        self.w = w


class _Exact:
    """The residual and what is built on it, on states of the valid cells
    (7 x N) in the grid file's order; every function is differentiable."""

    def __init__(self, c, g=None, cfg=None):
        if g is None:
            g, cfg = _grid_and_config(c)
        self.c, self.g, self.cfg, self.m = c, g, cfg, _Mesh(g, cfg)
        self.gas, self.tp = cfg.gas, cfg.transport

    def ghosts(self, s, when, sg):
        """Ghost rows (7 x G) after the actions of one list."""
        m, rows = self.m, []
        for name, f, valid, ids in m.tags:
            v = s[:, valid]
            q = sg[:, ids - m.N] if sg is not None else torch.zeros_like(v)
            for act in getattr(self.cfg.boundaries[name], when):
                kind = act["type"]
                if kind == "flow_state_copy":
                    fs = act["flow_state"]
                    q = torch.tensor([fs[k] for k in ("rho", "p", "T", "energy", "vx", "vy", "vz")],
                                     dtype=F64, device=DEV)[:, None].expand_as(v)
                elif kind == "internal_copy":
                    q = v
                elif kind == "internal_copy_reflect_normal":
                    vn = (v[VX:] * m.n[f].T).sum(dim=0)
                    q = torch.cat([v[:VX], v[VX:] - 2.0 * vn * m.n[f].T])
                elif kind == "internal_vel_copy_reflect":
                    q = torch.cat([q[:VX], -v[VX:]])
                elif kind == "fix_temperature":
                    q = torch.cat([q[:T], 2.0 * act["temperature"] - v[T:T + 1], q[E:]])
                else:
                    raise ValueError(kind)
            rows.append(q)
        return torch.cat(rows, dim=1)

    def gradient(self, u):
        m = self.m
        return ((u[m.nbr] - u[:m.N, None])[..., None] * m.w).sum(dim=1)

    def limiter(self, u, grad, d):
        m, kind = self.m, self.c["limiter"]
        ui, un = u[:m.N], u[m.nbr]
        hi, lo = ui, ui
        for j in range(un.shape[1]):
            hi, lo = torch.maximum(hi, un[:, j]), torch.minimum(lo, un[:, j])
        d2 = (grad[:, None] * d).sum(dim=2)
        up, down = d2 > 0, d2 < 0
        d1 = torch.where(up, (hi - ui)[:, None], (lo - ui)[:, None])
        if kind == "barth_jespersen":
            eps = self.cfg.epsilon
            den = torch.where(up, d2 + eps, torch.where(down, d2 - eps, torch.ones_like(d2)))
            ratio = d1 / den
        else:
            V = m.vol.abs()
            K3 = self.cfg.venkat_K ** 3
            eps2 = (K3 * V if m.dim == 3 else K3 * V * torch.sqrt(V))[:, None]
            num = d1 * d1 + eps2 + 2.0 * d1 * d2
            den = d1 * d1 + 2.0 * d2 * d2 + d1 * d2 + eps2
            ratio = num / den
        ratio = torch.where(up | down, ratio, torch.ones_like(ratio))
        return torch.clamp(ratio.min(dim=1).values, max=1.0)

    def closure(self, a, b):
        R, Cv, kind = self.gas.R, self.gas.Cv, self.c["thermo"]
        if kind == "rho_p":
            p, rho = a, b
            temp = p / (rho * R)
        elif kind == "rho_T":
            rho, temp = a, b
            p = rho * R * temp
        elif kind == "rho_u":
            rho, temp = a, b / Cv
            p = rho * R * temp
        else:
            p, temp = a, b
            rho = p / (R * temp)
        return rho, p, temp

    def flux(self, left, right):
        """Face-frame fluxes of (rho, p, T, u, v, w) on either side."""
        R, Cv, gamma = self.gas.R, self.gas.Cv, self.gas.gamma
        (rL, pL, TL, uL, vL, wL), (rR, pR, TR, uR, vR, wR) = left, right
        aL, aR = torch.sqrt(gamma * R * TL), torch.sqrt(gamma * R * TR)
        HL = Cv * TL + pL / rL + 0.5 * (uL * uL + vL * vL + wL * wL)
        HR = Cv * TR + pR / rR + 0.5 * (uR * uR + vR * vR + wR * wR)
        W, one = torch.where, torch.ones_like(rL)
        kind = self.c["flux"]
        if kind == "rusanov":
            S = torch.maximum(torch.maximum((uL - aL).abs(), (uR - aR).abs()),
                              torch.maximum((uL + aL).abs(), (uR + aR).abs()))
            qL, qR = (rL, rL * uL, rL * vL, rL * wL, rL * HL), (rR, rR * uR, rR * vR, rR * wR, rR * HR)
            out = [0.5 * (a * uL + b * uR) - 0.5 * S * (b - a) for a, b in zip(qL, qR)]
            out[1] = out[1] + 0.5 * (pL + pR)
            return out
        if kind == "hanel":
            subL, subR = uL.abs() <= aL, uR.abs() <= aR
            uLs, uRs = W(subL, one, uL), W(subR, one, uR)
            up = W(subL, (uL + aL) ** 2 / (4.0 * aL), 0.5 * (uL + uL.abs()))
            um = W(subR, -(uR - aR) ** 2 / (4.0 * aR), 0.5 * (uR - uR.abs()))
            pp = pL * up * W(subL, (2.0 - uL / aL) / aL, 1.0 / uLs)
            pm = pR * um * W(subR, (-2.0 - uR / aR) / aR, 1.0 / uRs)
            mL, mR = up * rL, um * rR
            return [mL + mR, mL * uL + mR * uR + pp + pm, mL * vL + mR * vR, mL * wL + mR * wR,
                    mL * HL + mR * HR]
        xL, xR = pL / rL, pR / rR
        alL, alR = 2.0 * xL / (xL + xR), 2.0 * xR / (xL + xR)
        am = torch.maximum(aL, aR)
        ML, MR = uL / am, uR / am
        subL, subR = ML.abs() <= 1.0, MR.abs() <= 1.0
        uLs, uRs = W(subL, one, uL), W(subR, one, uR)
        duL, duR = 0.5 * (uL + uL.abs()), 0.5 * (uR - uR.abs())
        pp = W(subL, pL * (ML + 1.0) ** 2 * (2.0 - ML) * 0.25, pL * duL / uLs)
        up = W(subL, alL * ((uL + am) ** 2 / (4.0 * am) - duL) + duL, duL)
        pm = W(subR, pR * (MR - 1.0) ** 2 * (2.0 + MR) * 0.25, pR * duR / uRs)
        um = W(subR, alR * (-(uR - am) ** 2 / (4.0 * am) - duR) + duR, duR)
        ru = up * rL + um * rR
        s = 0.5 * torch.clamp(10.0 * (pL - pR).abs() / torch.minimum(pL, pR), max=1.0)
        vv = up * rL * uL + um * rR * uR
        dd = 0.5 * (ru * (uL + uR) - ru.abs() * (uR - uL))
        pos = ru >= 0.0
        out = [ru, (0.5 + s) * vv + (0.5 - s) * dd + pp + pm, ru * W(pos, vL, vR),
               ru * W(pos, wL, wR), ru * W(pos, HL, HR)]
        caseA = ((uL - aL) < 0) & ((uR - aR) > 0)
        caseB = ((uL + aL) < 0) & ((uR + aR) > 0)
        fix = W(caseA & ~caseB, (uR - aR) - (uL - aL),
                W(caseB & ~caseA, (uR + aR) - (uL + aL), torch.zeros_like(rL))) * 0.125
        qL, qR = (rL, rL * uL, rL * vL, rL * wL, rL * HL), (rR, rR * uR, rR * vR, rR * wR, rR * HR)
        return [o - fix * (b - a) for o, a, b in zip(out, qL, qR)]

    def face_flux(self, s, recon=True, frozen=False):
        """(dim+2) x F fluxes in the global frame, the face states of the time
        step (density, T; None when inviscid) and the ghost rows."""
        m = self.m
        sg = self.ghosts(s, "pre_reconstruction", None)
        U = torch.cat([s, sg], dim=1)
        pair = {"rho_p": (P, RHO), "rho_T": (RHO, T), "rho_u": (RHO, E), "p_T": (P, T)}[self.c["thermo"]]
        sides = [[], []]
        if recon:
            d = m.xf[m.cell_faces] - m.xc[:m.N, None]
            for k, row in enumerate((*pair, VX, VY, VZ)):
                u = U[row]
                if m.dim == 2 and row == VZ:  # no vz gradient is computed in 2D
                    for q, c in enumerate((m.L, m.R)):
                        sides[q].append(u[c])
                    continue
                grad = self.gradient(u)
                phi = self.limiter(u, grad, d)
                slope = (phi.detach() if frozen else phi)[:, None] * grad
                slope = torch.cat([slope, slope.new_zeros((m.Nt - m.N, 3))])
                for q, c in enumerate((m.L, m.R)):
                    sides[q].append(u[c] + (slope[c] * (m.xf - m.xc[c])).sum(dim=1))
            states = [self.closure(x[0], x[1]) + tuple(x[2:]) for x in sides]
        else:
            states = [(U[RHO, c], U[P, c], U[T, c], U[VX, c], U[VY, c], U[VZ, c])
                      for c in (m.L, m.R)]
        frame = (m.n, m.t1, m.t2)
        local = []
        for rho, p, temp, a, b, cc in states:
            local.append((rho, p, temp, *[a * e[:, 0] + b * e[:, 1] + cc * e[:, 2] for e in frame]))
        f = self.flux(*local)
        rows = [f[0]] + [f[1] * m.n[:, k] + f[2] * m.t1[:, k] + (f[3] * m.t2[:, k] if m.dim == 3 else 0.0)
                         for k in range(m.dim)] + [f[4]]
        out, rho_f, T_f = torch.stack(rows), None, None
        if self.cfg.viscous:
            sg = self.ghosts(s, "pre_viscous_grad", sg)
            U = torch.cat([s, sg], dim=1)
            tau, rho_f, T_f = self.viscous(U)
            out = torch.cat([out[:1], out[1:] - tau])
        return out, rho_f, T_f, sg

    def viscosity(self, temp):
        tp = self.tp
        return tp.mu0 * (temp / tp.T0) * torch.sqrt(temp / tp.T0) * (tp.T0 + tp.Ts) / (temp + tp.Ts)

    def viscous(self, U):
        m = self.m
        L, R = m.L, m.R
        inner = (L < m.N) & (R < m.N)
        valid = torch.where(L < m.N, L, R)
        e = m.xc[R] - m.xc[L]
        length = _norm(e)
        ehat = e / length[:, None]
        edn = (ehat * m.n).sum(dim=1)
        g = {}
        for row in (T, VX, VY, VZ):
            grad = self.gradient(U[row])
            pad = torch.cat([grad, grad.new_zeros((m.Nt - m.N, 3))])
            avg = 0.5 * (pad[L] + pad[R])
            corr = (avg * ehat).sum(dim=1) - (U[row, R] - U[row, L]) / length
            g[row] = torch.where(inner[:, None], avg - (corr / edn)[:, None] * m.n, pad[valid])
        mid = {row: 0.5 * (U[row, L] + U[row, R]) for row in (P, T, VX, VY, VZ)}
        mu = self.viscosity(mid[T])
        k = self.gas.Cp * mu / self.tp.Pr
        v = [g[VX], g[VY], g[VZ]]
        div = v[0][:, 0] + v[1][:, 1] + v[2][:, 2]
        tau = [[mu * (v[a][:, b] + v[b][:, a]) - ((2.0 / 3.0) * mu * div if a == b else 0.0)
                for b in range(3)] for a in range(3)]
        vel = (mid[VX], mid[VY], mid[VZ])
        rows = [sum(m.n[:, b] * tau[a][b] for b in range(3)) for a in range(m.dim)]
        theta = [sum(vel[a] * tau[a][b] for a in range(3)) + k * g[T][:, b] for b in range(3)]
        rows.append(sum(m.n[:, b] * theta[b] for b in range(3)))
        return torch.stack(rows), mid[P] / (self.gas.R * mid[T]), mid[T]

    def residual(self, s, recon=True, frozen=False):
        m = self.m
        f, rho_f, T_f, sg = self.face_flux(s, recon, frozen)
        fa = f * m.area
        d = -(fa[:, m.cell_faces] * m.sign).sum(dim=2) / m.vol
        return d, f, (rho_f, T_f), sg

    def force(self, f, tag):
        m = self.m
        total = 0.0
        for name, faces, _, _ in m.tags:
            if name == tag:
                s = torch.where(m.L[faces] < m.N, m.area[faces], -m.area[faces])
                total = total + sum(_FORCE_DIR[k] * (f[1 + k, faces] * s).sum() for k in range(m.dim))
        return total

    def dt(self, s, face):
        m, gas = self.m, self.gas
        cf = m.cell_faces
        a = torch.sqrt(gas.gamma * gas.R * s[T])
        vn = (s[VX:].T[:, None] * m.n[cf]).sum(dim=2)
        rate = ((vn.abs() + a[:, None]) * m.area[cf]).sum(dim=1)
        if face[0] is not None:
            mu = self.viscosity(face[1])
            # mu / Pr with Pr = mu Cp / k, k = Cp mu / Pr
            x = gas.gamma / face[0] * mu / self.tp.Pr * m.area ** 2
            rate = rate + self.cfg.signal_factor * x[cf].sum(dim=1) / m.vol
        return float((m.vol / rate).min())

    def prim(self, q):
        gas, dim = self.gas, self.m.dim
        rho = q[0]
        v = [q[1 + k] / rho for k in range(dim)]
        if dim == 2:
            v.append(torch.zeros_like(rho))
        u = q[dim + 1] / rho - 0.5 * (v[0] * v[0] + v[1] * v[1] + v[2] * v[2])
        temp = u / gas.Cv
        return torch.stack([rho, rho * gas.R * temp, temp, u, *v])

    def rk3(self, q, s, dt_prev):
        """One ssp-rk3 step of the valid cells: conserved, primitive, dt."""
        k1, _, face, _ = self.residual(s)
        dt = min(0.5 * self.dt(s, face), 1.5 * dt_prev)
        k2 = self.residual(self.prim(q + dt * k1))[0]
        k3 = self.residual(self.prim(q + 0.25 * dt * (k1 + k2)))[0]
        q = q + dt / 6.0 * (k1 + k2 + 4.0 * k3)
        return q, self.prim(q), dt

    def matvec(self, q, v, dt_star, recon=True):
        """vec / dt* - (dR/dU) vec on (dim+2) x N arrays."""
        jv = torch.func.jvp(lambda x: self.residual(self.prim(x), recon)[0], (q,), (v,))[1]
        return v / dt_star - jv

    def gmres(self, A, rhs, iters, tol, inner=None):
        """x from zero, and the number of iterations."""
        beta = float(rhs.norm())
        V, Z, H = [rhs / beta], [], np.zeros((iters + 1, iters))
        for j in range(iters):
            Z.append(inner(V[j]) if inner else V[j])
            w = A(Z[j])
            for i in range(j + 1):
                H[i, j] = float((w * V[i]).sum())
                w = w - H[i, j] * V[i]
            H[j + 1, j] = float(w.norm())
            V.append(w / H[j + 1, j])
            e = np.zeros(j + 2)
            e[0] = beta
            y = np.linalg.lstsq(H[:j + 2, :j + 1], e, rcond=None)[0]
            if np.linalg.norm(H[:j + 2, :j + 1] @ y - e) < tol * beta:
                break
        return sum(float(y[i]) * Z[i] for i in range(len(y))), len(y)


def _out(a, n_total, order, ghosts=None):
    """(rows, N) of the grid file's order as (rows, N_total) of the grid's."""
    full = a.new_zeros((a.shape[0], n_total))
    full[:, :a.shape[1]] = a
    if ghosts is not None:
        full[:, a.shape[1]:] = ghosts
    return _ordered(full, order)


def exact(case, seed):
    c, what = case, case["what"]
    if what == "batch":
        return _exact_batch(c, seed)
    g, cfg = _grid_and_config(c)
    x = _Exact(c, g, cfg)
    N, Nt, dim = x.m.N, x.m.Nt, x.m.dim
    order = torch.from_numpy(GridBlock(g, cfg, reorder=True, device=False).cell_new_of_old).to(DEV)
    full = _state(c, g, Nt - N, seed)
    s, g0 = full[:, :N].contiguous(), full[:, N:]
    put = lambda a, gh=None: _out(a, Nt, order, gh)  # noqa: E731
    if what == "residual":
        d, _, _, sg = x.residual(s)
        return {"dudt": put(d), "prim": put(s, sg)}
    if what == "rk":
        q, s, dt = x.rk3(_cons(s, dim), s, math.inf)
        gq = _cons(g0, dim)
        return {"cons": put(q, gq), "prim": put(s, x.prim(gq)), "dt": dt}
    if what in ("vjp", "autograd"):
        bar = _vector(c, g, Nt - N, seed)[1][:, :N]
        s.requires_grad_(True)
        d, f, _, sg = x.residual(s, frozen=c["mode"] == "frozen")
        j = x.force(f, _force_tag(c))
        (grad,) = torch.autograd.grad((d * bar).sum() + j, s)
        s = s.detach()
        if what == "vjp":
            return {"prim_bar": put(grad), "prim": put(s, sg.detach())}
        return {"dudt": put(d.detach()), "force": j.detach(), "grad": put(grad)}
    if what == "jvp":
        dot = _vector(c, g, Nt - N, seed)[0][:, :N]

        def both(v):
            d, _, _, sg = x.residual(v)
            return d, sg
        (d, sg), (dd, sgd) = torch.func.jvp(both, (s,), (dot,))
        return {"dudt": put(d), "dudt_dot": put(dd), "prim": put(s, sg), "dot": put(dot, sgd)}
    q = _cons(s, dim)
    if what == "matvec":
        dot = _vector(c, g, Nt - N, seed)[0][:, :N]
        v = torch.func.jvp(lambda y: _cons(y, dim), (s,), (dot,))[1]
        return {"result": _cell_major(put(x.matvec(q, v, _DT_STAR)), N)}
    d, _, face, _ = x.residual(s)
    dt_star = c["cfl"] * x.dt(s, face)
    inner = None
    if c["solver"] == "fgmres":
        P1 = lambda v: x.matvec(q, v, dt_star, recon=False)  # noqa: E731
        inner = lambda v: x.gmres(P1, v, c["inner_iters"], c["inner_tol"])[0]  # noqa: E731
    du, iters = x.gmres(lambda v: x.matvec(q, v, dt_star), d, c["iters"], c["tol"], inner)
    q = q + du
    s = x.prim(q)
    d, _, _, sg = x.residual(s)
    rows = [d[0], d[1], d[2], d[3] if dim == 3 else torch.zeros_like(d[0]), d[dim + 1]]
    norms = [float(r.norm()) for r in rows] + [float(d.norm())]
    return {"cons": put(q, _cons(g0, dim)), "prim": put(s, sg), "iters": iters, "norms": norms}


def _exact_batch(c, seed):
    cons, prim = [], []
    for k, i in enumerate(_instances(c)):
        g, cfg = _grid_and_config(i)
        x = _Exact(i, g, cfg)
        N, Nt = x.m.N, x.m.Nt
        order = torch.from_numpy(GridBlock(g, cfg, reorder=True, device=False).cell_new_of_old).to(DEV)
        full = _state(i, g, Nt - N, seed + 100 * k)
        s, q, dt = full[:, :N], _cons(full[:, :N], 2), math.inf
        for _ in range(c["steps"]):
            q, s, dt = x.rk3(q, s, dt)
        gq = _cons(full[:, N:], 2)
        cons.append((_out(q, Nt, order, gq), N))
        prim.append((_out(s, Nt, order, x.prim(gq)), N))
    join = lambda parts: torch.cat([a[:, :n] for a, n in parts] +  # noqa: E731
                                   [a[:, n:] for a, n in parts], dim=1)
    return {"cons": join(cons), "prim": join(prim)}
