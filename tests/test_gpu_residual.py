"""Parity of the MI355X residual with the oracle (run on the GPU box).

Inviscid residuals compare bit for bit: the kernels and the oracle evaluate
the same IEEE expression trees with contraction disabled.  Viscous and
LDFSS2 residuals go through pow() (Sutherland, LDFSS2), where the device and
host math libraries may differ in the last bit, so they are compared at
1e-12 relative per conserved variable (max |gpu - cpu| / max |cpu|).
"""
import numpy as np
import pytest

from helpers import gpu_dudt, gpu_objects, oracle_pair, rel_err, to_dev
from ibis_amd import cases

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _check(grid_io, cfg, prim_ref, exact, allow_reconstruction=True, options=None):
    og, ofv = oracle_pair(grid_io, cfg)
    p_cpu = prim_ref.copy()
    d_cpu = ofv.compute_dudt(p_cpu, allow_reconstruction=allow_reconstruction)
    gb, fv = gpu_objects(grid_io, cfg)
    for k, v in (options or {}).items():
        fv.set_option(k, v)
    d_gpu, p_gpu = gpu_dudt(gb, fv, prim_ref, allow_reconstruction)
    n = og.N
    print(f"case N={n} F={og.F} flux={cfg.flux} lim={cfg.limiter} visc={cfg.viscous}", flush=True)
    assert np.isfinite(d_cpu[:, :n]).all()
    if exact:
        assert np.array_equal(d_gpu[:, :n], d_cpu[:, :n]), rel_err(d_gpu, d_cpu, n)
    else:
        err = rel_err(d_gpu, d_cpu, n)
        assert (err <= TOL).all(), err
    # ghost rows written by the boundary actions (bit-exact in all cases)
    assert np.array_equal(p_gpu[:, n:], p_cpu[:, n:])
    # time step
    dt_cpu = ofv.estimate_dt(p_cpu)
    dt_gpu = fv.estimate_dt(to_dev(gb.to_grid_order(p_cpu)))
    if exact:
        assert dt_gpu == dt_cpu
    else:
        assert abs(dt_gpu - dt_cpu) <= TOL * dt_cpu
    return og, ofv, gb, fv


WEDGE_VARIANTS = [
    dict(flux="ausmdv", limiter="barth_jespersen", thermo="rho_u"),
    dict(flux="hanel", limiter="barth_jespersen", thermo="rho_u"),
    dict(flux="rusanov", limiter="barth_jespersen", thermo="rho_u"),
    dict(flux="ausmdv", limiter="unlimited", thermo="rho_u"),
    dict(flux="ausmdv", limiter="venkatakrishnan", thermo="rho_u"),
    dict(flux="ausmdv", limiter="barth_jespersen", thermo="rho_p"),
    dict(flux="ausmdv", limiter="barth_jespersen", thermo="rho_T"),
    dict(flux="hanel", limiter="barth_jespersen", thermo="p_T"),
    dict(flux="ausmdv", limiter="barth_jespersen", thermo="rho_u", order=1),
]


@pytest.mark.parametrize("kw", WEDGE_VARIANTS, ids=lambda k: "-".join(str(v) for v in k.values()))
def test_wedge_variants(kw):
    g_io, cfg, fs = cases.wedge_case(48, 24, **kw)
    prim = cases.perturbed_prim(g_io, fs, g_io.num_cells + 2 * (48 + 24), seed=11)
    _check(g_io, cfg, prim, exact=True)


@pytest.mark.parametrize("layout", [0, 2])
def test_wedge_subsonic_boundaries(layout):
    """Subsonic inflow / outflow and slip-wall actions on the second-order
    inviscid path: boundary actions fused with the ghost face values (layout
    0), and run in the cell kernel's staging of each ghost (layout 2, the
    option fold_boundary) or as a kernel of their own (fold_boundary 0)."""
    from ibis_amd import config as C
    g_io, cfg, fs = cases.wedge_case(48, 24, mach=0.5)
    cfg.boundaries = {"inflow": C.subsonic_inflow(fs), "outflow": C.subsonic_outflow(fs.p * 0.98),
                      "wall": C.slip_wall()}
    prim = cases.perturbed_prim(g_io, fs, g_io.num_cells + 2 * (48 + 24), seed=15)
    _check(g_io, cfg, prim, exact=True, options={"face_state_layout": layout})
    if layout == 2:
        _check(g_io, cfg, prim, exact=True, options={"fold_boundary": 0})


@pytest.mark.parametrize("zmode", ["flat", "uneven"])
def test_2d_mesh_off_the_z0_plane(zmode):
    """A 2D wedge lifted to z = 1.5 (every centroid at the same z: the 2D
    kernels take each z difference as +0 without loading it) and one whose
    vertices' z differ (they load it): the fused inviscid residual with and
    without precomputed offsets bit for bit, and the fused viscous one at the
    viscous bar, against the oracle."""
    from ibis_amd import config as C
    from ibis_amd import gridgen

    def lift(g_io):
        if zmode == "flat":
            g_io.xyz[:, 2] = 1.5
        else:
            g_io.xyz[:, 2] = 1.5 + 1e-3 * gridgen.uniform01(17, g_io.xyz.shape[0])
        return g_io

    g_io, cfg, fs = cases.wedge_case(40, 20)
    g_io = lift(g_io)
    prim = cases.perturbed_prim(g_io, fs, 40 * 20 + 2 * (40 + 20), seed=23)
    print(f"2D off z=0: {zmode}", flush=True)
    _check(g_io, cfg, prim, exact=True)
    _check(g_io, cfg, prim, exact=True, options={"precomputed_offsets": 0})
    g_io, cfg, fs = cases.wedge_case(40, 20, mach=0.5)
    g_io = lift(g_io)
    cfg.viscous = True
    cfg.boundaries = {"inflow": C.subsonic_inflow(fs), "outflow": C.subsonic_outflow(fs.p * 0.98),
                      "wall": C.fixed_temperature_no_slip_wall(300.0)}
    _check(g_io, cfg, cases.perturbed_prim(g_io, fs, 40 * 20 + 2 * 60, seed=24), exact=False)


def test_wedge_ldfss2_tolerance():
    g_io, cfg, fs = cases.wedge_case(48, 24, flux="ldfss2")
    prim = cases.perturbed_prim(g_io, fs, g_io.num_cells + 2 * (48 + 24), seed=12)
    _check(g_io, cfg, prim, exact=False)


def test_wedge_first_order_when_reconstruction_disallowed():
    g_io, cfg, fs = cases.wedge_case(48, 24)
    prim = cases.perturbed_prim(g_io, fs, g_io.num_cells + 2 * (48 + 24), seed=13)
    _check(g_io, cfg, prim, exact=True, allow_reconstruction=False)


def test_wedge_192x96_full_size():
    """192 x 96 wedge, AUSMDV / Barth-Jespersen / rho_u, uniform Mach 3 and
    perturbed states."""
    g_io, cfg, fs = cases.wedge_case(192, 96)
    nt = g_io.num_cells + 2 * (192 + 96)
    _check(g_io, cfg, cases.uniform_prim(fs, g_io.num_cells, nt), exact=True)
    _check(g_io, cfg, cases.perturbed_prim(g_io, fs, nt, seed=14), exact=True)


@pytest.mark.parametrize("flux,limiter", [("hanel", "venkatakrishnan"),
                                          ("ausmdv", "barth_jespersen"),
                                          ("rusanov", "unlimited")])
def test_hex_jittered_permuted(flux, limiter):
    g_io, cfg = cases.hex_case(16, flux=flux, limiter=limiter)
    prim = cases.hex_prim(g_io, 16 ** 3 + 6 * 16 ** 2)
    _check(g_io, cfg, prim, exact=True)


@pytest.mark.parametrize("layout,pack,fk,stage,pf,sc", [(0, 1, 0, 1, 0, 0), (1, 1, 0, 0, 0, 0),
                                                         (2, 1, 0, 1, 0, 0), (2, 0, 0, 1, 0, 0),
                                                         (2, 0, 0, 0, 1, 0), (2, 1, 64, 0, 0, 0),
                                                         (2, 0, 1, 1, 1, 0), (2, 1, 1, 0, 0, 0),
                                                         (2, 0, 128, 1, 1, 0), (2, 1, 256, 1, 0, 0),
                                                         (2, 0, 1, 1, 0, 1), (2, 0, 0, 0, 1, 1)])
@pytest.mark.parametrize("offsets", [0, 1])
def test_implementation_options_give_identical_bits(layout, pack, fk, stage, pf, sc, offsets):
    opts = {"face_state_layout": layout, "precomputed_offsets": offsets, "pack_cells": pack,
            "face_kernel": fk, "stage_offsets": stage, "cell_prefetch": pf, "stage_cells": sc}
    g_io, cfg = cases.hex_case(12, flux="hanel", limiter="venkatakrishnan")
    _check(g_io, cfg, cases.hex_prim(g_io, 12 ** 3 + 6 * 12 ** 2), exact=True, options=opts)
    g_io, cfg, fs = cases.wedge_case(40, 20)
    prim = cases.perturbed_prim(g_io, fs, 40 * 20 + 2 * (40 + 20), seed=21)
    _check(g_io, cfg, prim, exact=True, options=opts)


TILE_OPTIONS = [{"tile": 128}, {"tile": 512}, {"fold_boundary": 0}, {"fold_boundary": 1},
                {"tile": 512, "face_kernel": 0}, {"tile": 128, "stage_cells": 0, "cell_prefetch": 1},
                {"tile": 512, "face_state_layout": 0, "pack_cells": 1, "face_kernel": 0}]


@pytest.mark.parametrize("opts", TILE_OPTIONS, ids=lambda o: "-".join(f"{k}{v}" for k, v in o.items()))
def test_tile_sizes_give_identical_bits(opts):
    """Tiles of 128 and 512 cells (the tile kernels' block size follows)
    on the 12^3 hex box, the wedge, the first-order wedge and the
    hex/pyramid mesh, bit for bit against the oracle."""
    from ibis_amd import gridgen
    g_io, cfg = cases.hex_case(12, flux="hanel", limiter="venkatakrishnan")
    _check(g_io, cfg, cases.hex_prim(g_io, 12 ** 3 + 6 * 12 ** 2), exact=True, options=opts)
    g_io, cfg, fs = cases.wedge_case(40, 20)
    prim = cases.perturbed_prim(g_io, fs, 40 * 20 + 2 * (40 + 20), seed=21)
    _check(g_io, cfg, prim, exact=True, options=opts)
    g_io, cfg, fs = cases.wedge_case(40, 20, order=1)
    _check(g_io, cfg, prim, exact=True, options=opts)
    g_io, cfg = cases.hex_case(8, flux="hanel", limiter="venkatakrishnan")
    gh = gridgen.split_hexes(g_io, 3)
    _check(gh, cfg, cases.hex_prim(gh, gh.num_cells + 6 * 64), exact=True, options=opts)


def test_tile_option_switches_on_one_residual():
    """One residual switched between tile sizes (512, 128, 256, 512) and to
    the FP32-flux mode and back: every FP64 residual equals the oracle's bit
    for bit, so the per-entry face data follows each switch."""
    g_io, cfg = cases.hex_case(10, flux="ausmdv", limiter="barth_jespersen")
    prim = cases.hex_prim(g_io, 10 ** 3 + 6 * 10 ** 2)
    og, ofv = oracle_pair(g_io, cfg)
    d_cpu = ofv.compute_dudt(prim.copy())
    gb, fv = gpu_objects(g_io, cfg)
    for tile in (512, 128, 256, 512):
        fv.set_option("tile", tile)
        fv.set_precision("fp32_flux")
        gpu_dudt(gb, fv, prim)
        fv.set_precision("fp64")
        d_gpu, _ = gpu_dudt(gb, fv, prim)
        print(f"tile {tile}", flush=True)
        assert np.array_equal(d_gpu[:, :og.N], d_cpu[:, :og.N]), tile


MIXED_OPTIONS = [{}, {"face_state_layout": 0, "face_kernel": 0, "stage_cells": 0,
                      "precomputed_offsets": 0, "pack_cells": 1},
                 {"stage_cells": 0, "cell_prefetch": 1, "face_kernel": 0},
                 {"face_kernel": 128, "stage_cells": 0}]


@pytest.mark.parametrize("opts", MIXED_OPTIONS, ids=["default", "layout0", "prefetch", "slot128"])
def test_mixed_elements_ragged_stencils(opts):
    """Cells with different face counts: a 2D triangle / quad mesh (3 and 4
    faces) and a 3D hex / pyramid mesh (5 and 6 faces, triangle and quad
    faces), bit for bit against the oracle."""
    from ibis_amd import gridgen
    g_io, cfg, fs = cases.wedge_case(24, 12)
    gm = gridgen.split_quads(g_io, 2)
    prim = cases.perturbed_prim(gm, fs, gm.num_cells + 2 * (24 + 12), seed=31)
    _check(gm, cfg, prim, exact=True, options=opts)
    g_io, cfg = cases.hex_case(8, flux="hanel", limiter="venkatakrishnan")
    gh = gridgen.split_hexes(g_io, 3)
    _check(gh, cfg, cases.hex_prim(gh, gh.num_cells + 6 * 64), exact=True, options=opts)


@pytest.mark.parametrize("case", ["wedge", "hex"])
def test_stored_normals_entry_kernel_matches_tile_kernel(case):
    """A caller's mesh whose normals are not exactly cross(t1, t2) keeps its
    stored normals.  The per-entry face kernel then loads them with the
    entry geometry; the tile-list kernel reads them from the face geometry.
    The two kernels must agree bit for bit, and the stored normals must be
    used (the residual differs from the unperturbed mesh's)."""
    import ctypes as C
    from types import SimpleNamespace

    import torch

    from ibis_amd.batch import _concat_grids
    from ibis_amd.finite_volume import FiniteVolume, GridBlock
    from ibis_amd.native import MeshDescStruct, check, lib, ptr

    if case == "wedge":
        g_io, cfg, fs = cases.wedge_case(32, 16)
        prim_ref = cases.perturbed_prim(g_io, fs, 32 * 16 + 2 * (32 + 16), seed=41)
    else:
        g_io, cfg = cases.hex_case(10, flux="hanel", limiter="venkatakrishnan")
        prim_ref = cases.hex_prim(g_io, 10 ** 3 + 6 * 10 ** 2)
    gb = GridBlock(g_io, cfg)
    arr, N, G, F, _, _ = _concat_grids([gb])
    geom = arr["face_geom"]
    geom[0, ::3] = np.nextafter(geom[0, ::3], np.inf)  # n_x of every third face, one ulp
    d = MeshDescStruct()
    d.dim, d.ntags = gb.dim, len(arr["tag_off"]) - 1
    d.n_cells, d.n_ghost, d.n_faces = N, G, F
    for k, v in arr.items():
        setattr(d, k, ptr(v))
    m = C.c_void_p()
    check(lib().ibis_mesh_create(C.byref(d), C.byref(m)), "ibis_mesh_create")
    fv = ref_fv = None
    try:
        mesh = SimpleNamespace(_mesh=m, dim=gb.dim, Nt=gb.Nt)
        fv = FiniteVolume(mesh, cfg)
        prim0 = to_dev(gb.to_grid_order(prim_ref))
        out = {}
        for fk in (1, 0):
            fv.set_option("face_state_layout", 2)
            fv.set_option("face_kernel", fk)
            prim = prim0.clone()
            dudt = torch.zeros((gb.dim + 2, gb.Nt), dtype=torch.float64, device="cuda")
            fv.compute_dudt(prim, None, dudt)
            torch.cuda.synchronize()
            out[fk] = dudt.cpu().numpy()[:, :N]
        print(f"stored normals {case}: N={N} F={F}", flush=True)
        assert np.array_equal(out[1], out[0])
        ref_fv = FiniteVolume(gb, cfg)
        d_ref, _ = gpu_dudt(gb, ref_fv, prim_ref)
        assert not np.array_equal(out[1], gb.to_grid_order(d_ref)[:, :N])
    finally:
        for h in (fv, ref_fv):
            if h is not None:
                h.close()
        lib().ibis_mesh_destroy(m)
        gb.close()


def test_plate_viscous():
    g_io, cfg, fs = cases.plate_case(64, 32)
    prim = cases.perturbed_prim(g_io, fs, 64 * 32 + 2 * (64 + 32), seed=2)
    _check(g_io, cfg, prim, exact=False)


@pytest.mark.timeout(300)
def test_plate_viscous_1024x512_full_size():
    g_io, cfg, fs = cases.plate_case(1024, 512)
    prim = cases.perturbed_prim(g_io, fs, 1024 * 512 + 2 * (1024 + 512), seed=2)
    _check(g_io, cfg, prim, exact=False)


def test_count_bad_cells():
    g_io, cfg, fs = cases.wedge_case(48, 24)
    nt = g_io.num_cells + 2 * (48 + 24)
    prim = cases.uniform_prim(fs, g_io.num_cells, nt)
    prim[2, 5] = -1.0          # T < 0
    prim[0, 17] = np.nan       # rho NaN
    prim[0, 100] = np.inf      # rho Inf
    prim[0, 7] = -2.0          # rho < 0
    og, ofv = oracle_pair(g_io, cfg)
    gb, fv = gpu_objects(g_io, cfg)
    assert ofv.count_bad_cells(prim) == 4
    assert fv.count_bad_cells(to_dev(gb.to_grid_order(prim))) == 4


def test_rk_steps_match_oracle():
    """Five ssp-rk3 steps at CFL 0.5 on the wedge: identical state and dt."""
    import torch
    from ibis_amd.config import ssp_rk3
    from ibis_amd.finite_volume import RungeKutta
    g_io, cfg, fs = cases.wedge_case(48, 24)
    nt = g_io.num_cells + 2 * (48 + 24)
    prim = cases.perturbed_prim(g_io, fs, nt, seed=15)
    og, ofv = oracle_pair(g_io, cfg)
    cons = ofv.prim_to_cons(prim)
    gb, fv = gpu_objects(g_io, cfg)
    d_prim = to_dev(gb.to_grid_order(prim))
    d_cons = to_dev(gb.to_grid_order(cons))
    rk = RungeKutta(fv, "ssp-rk3", cfl=0.5, max_time=1.0)
    a, b = ssp_rk3()
    dt_prev, t = np.finfo(np.float64).max, 0.0
    p_cpu, c_cpu = prim.copy(), cons.copy()
    for step in range(5):
        dt_cpu = ofv.rk_step(a, b, 0.5, c_cpu, p_cpu, dt_prev, t, 1.0)
        dt_prev = dt_cpu
        t += dt_cpu
        dt_gpu = rk.take_step(d_cons, d_prim)
        assert dt_gpu == dt_cpu
    torch.cuda.synchronize()
    c_gpu = gb.to_reference_order(d_cons.cpu().numpy())
    n = og.N
    assert np.array_equal(c_gpu[:, :n], c_cpu[:, :n])


@pytest.mark.timeout(900)
def test_wedge_192x96_2000_steps():
    """The 192 x 96 wedge workload: uniform Mach-3 free
    stream, ssp-rk3 at CFL 0.5, 2000 steps.  The plain path (a host dt per
    step) equals the oracle's state after steps 1, 10, 100 and 2000 and its
    dt at every step; the device-resident path (a batch of one, each step
    one HIP graph replay) equals it after 2000 steps."""
    import torch
    from ibis_amd.batch import Batch
    from ibis_amd.config import ssp_rk3
    from ibis_amd.finite_volume import RungeKutta
    from ibis_amd.native import check, lib, ptr
    g_io, cfg, fs = cases.wedge_case(192, 96)
    n = g_io.num_cells
    prim = cases.uniform_prim(fs, n, n + 2 * (192 + 96))
    og, ofv = oracle_pair(g_io, cfg)
    cons = ofv.prim_to_cons(prim)
    gb, fv = gpu_objects(g_io, cfg)
    d_prim, d_cons = to_dev(gb.to_grid_order(prim)), to_dev(gb.to_grid_order(cons))
    rk = RungeKutta(fv, "ssp-rk3", cfl=0.5, max_time=1e30)
    a, b = ssp_rk3()
    dt_prev, t = np.finfo(np.float64).max, 0.0
    p_cpu, c_cpu = prim.copy(), cons.copy()
    for step in range(1, 2001):
        dt_cpu = ofv.rk_step(a, b, 0.5, c_cpu, p_cpu, dt_prev, t, 1e30)
        dt_prev = dt_cpu
        t += dt_cpu
        assert rk.take_step(d_cons, d_prim) == dt_cpu, step
        if step in (1, 10, 100, 2000):
            torch.cuda.synchronize()
            c_gpu = gb.to_reference_order(d_cons.cpu().numpy())
            assert np.array_equal(c_gpu[:, :n], c_cpu[:, :n]), step
            print(f"wedge 192x96: step {step}, t = {t:.6e}, state identical to the oracle", flush=True)
    bt = Batch([(g_io, cfg)])
    b0 = bt.blocks[0]
    bp = to_dev(bt.gather([b0.to_grid_order(prim)]))
    bc = torch.zeros((bt.ncons, bt.Nt), dtype=torch.float64, device="cuda")
    check(lib().ibis_prim_to_cons(bt.residual_handle(), ptr(bp), ptr(bc), None), "prim_to_cons")
    bt.rk_init(bc, bp, cfl=0.5, max_time=1e30)
    bt.rk_steps(2000, use_graph=True)
    c_bat = b0.to_reference_order(bt.scatter(bc.cpu().numpy(), 0))
    assert np.array_equal(c_bat[:, :n], c_cpu[:, :n])
    tb, _ = bt.times()
    assert tb[0] == t
    bt.close()


@pytest.mark.timeout(600)
def test_renumbering_invariance_hex160():
    """Config-3 size (160^3 jittered, cell-permuted hexes): the residual on
    the locality-renumbered grid equals the residual on the reference
    numbering, bit for bit."""
    import torch
    g_io, cfg = cases.hex_case(160)
    nt = 160 ** 3 + 6 * 160 ** 2
    prim = cases.hex_prim(g_io, nt)
    outs = []
    for reorder in (True, False):
        print(f"hex160 reorder={reorder}: building grid", flush=True)
        gb, fv = gpu_objects(g_io, cfg, reorder=reorder)
        print("  residual", flush=True)
        d, _ = gpu_dudt(gb, fv, prim)
        outs.append(d)
        del fv, gb
        torch.cuda.empty_cache()
    n = 160 ** 3
    assert np.array_equal(outs[0][:, :n], outs[1][:, :n])
    assert np.isfinite(outs[0][:, :n]).all()


def _visc_cases():
    """Viscous cases for the fused viscous path: the plate (AUSMDV,
    Barth-Jespersen, fixed-temperature no-slip wall), the same with Hanel and
    Venkatakrishnan and rho_p, a split-quad plate (triangles and quads),
    a jittered permuted 3D box with slip and no-slip walls, and a subsonic
    wedge with viscous walls."""
    from ibis_amd import config as C
    from ibis_amd import gridgen
    out = {}
    g_io, cfg, fs = cases.plate_case(64, 32)
    out["plate"] = (g_io, cfg, cases.perturbed_prim(g_io, fs, 64 * 32 + 2 * (64 + 32), seed=2))
    g_io, cfg, fs = cases.plate_case(48, 24, flux="hanel")
    cfg.limiter, cfg.thermo_interpolator = "venkatakrishnan", "rho_p"
    out["plate_hanel_vk"] = (g_io, cfg, cases.perturbed_prim(g_io, fs, 48 * 24 + 2 * 72, seed=3))
    gm = gridgen.split_quads(g_io, 2)
    out["plate_triquad"] = (gm, cfg, cases.perturbed_prim(gm, fs, gm.num_cells + 2 * 72, seed=4))
    g_io, cfg = cases.hex_case(10, flux="ausmdv", limiter="barth_jespersen")
    cfg.viscous = True
    tags = sorted(cfg.boundaries)
    cfg.boundaries[tags[0]] = C.fixed_temperature_no_slip_wall(320.0)
    cfg.boundaries[tags[1]] = C.slip_wall()
    prim = cases.hex_prim(g_io, 10 ** 3 + 6 * 10 ** 2)
    prim[:, 10 ** 3:] = prim[:, :1]
    out["hex_walls"] = (g_io, cfg, prim)
    g_io, cfg, fs = cases.wedge_case(48, 24, mach=0.5)
    cfg.viscous = True
    cfg.boundaries = {"inflow": C.subsonic_inflow(fs), "outflow": C.subsonic_outflow(fs.p * 0.98),
                      "wall": C.fixed_temperature_no_slip_wall(300.0)}
    out["wedge_subsonic"] = (g_io, cfg, cases.perturbed_prim(g_io, fs, 48 * 24 + 2 * 72, seed=5))
    return out


@pytest.mark.parametrize("name", ["plate", "plate_hanel_vk", "plate_triquad", "hex_walls",
                                  "wedge_subsonic"])
def test_fused_viscous_path_equals_general_path(name):
    """The four-kernel viscous path (boundary actions, cell kernel with the
    viscous gradients, viscous terms per face, face kernel with the viscous
    flux) against the
    reference-shaped general path on the same device: dU/dt, the ghost rows,
    estimate_dt (face density and temperature) and, with keep_gradients,
    every gradient and limiter slot, bit for bit; and against the oracle at
    the viscous bar."""
    import torch
    g_io, cfg, prim_ref = _visc_cases()[name]
    _check(g_io, cfg, prim_ref, exact=False)
    gb, fv = gpu_objects(g_io, cfg)
    outs = []
    # the fused path with its boundary passes folded into the cell kernel's
    # staging (the default) and as a kernel of their own, then the general path
    for fuse, fold in ((1, 1), (1, 0), (0, 1)):
        fv.set_option("fuse_viscous", fuse)
        fv.set_option("fold_boundary", fold)
        fv.set_option("keep_gradients", 1)
        d, p = gpu_dudt(gb, fv, prim_ref)
        dt = fv.estimate_dt(to_dev(gb.to_grid_order(p)))
        grads = fv.cell_gradients().cpu().numpy()
        torch.cuda.synchronize()
        outs.append((d, p, dt, grads))
    n = gb.N
    print(f"{name}: N={n}", flush=True)
    for o in outs[:2]:
        assert o[0][:, :n].tobytes() == outs[2][0][:, :n].tobytes()
        assert o[1].tobytes() == outs[2][1].tobytes()
        assert o[2] == outs[2][2]
        assert o[3].tobytes() == outs[2][3].tobytes()


@pytest.mark.parametrize("method", ["euler", "midpoint", "ssp-rk3", "rk3", "rk4"])
@pytest.mark.parametrize("kind", ["wedge", "wedge_order1", "plate", "hex"])
def test_rk_step_equals_its_operations(kind, method):
    """ibis_rk_step (stage updates in the face kernel's epilogue, or one kernel
    a stage; the time step on the device) against the same step made of the
    library's single operations, bit for bit, ghost rows included, over three
    steps whose time step is the growth limit's, the CFL's and the end time's."""
    import torch
    from ibis_amd.config import butcher
    from ibis_amd.finite_volume import RungeKutta
    from ibis_amd.native import check, lib, ptr
    if kind == "hex":
        g_io, cfg = cases.gridgen.hex_box(7, jitter=0.0), cases.hex_config()
        ref = cases.hex_prim(g_io, 7 ** 3 + 6 * 49)
    else:
        make = cases.plate_case if kind == "plate" else cases.wedge_case
        g_io, cfg, fs = make(37, 19, **({"order": 1} if kind == "wedge_order1" else {}))
        ref = cases.perturbed_prim(g_io, fs, 37 * 19 + 2 * (37 + 19), seed=91)
    ref[:, g_io.num_cells:] = ref[:, :1]
    out = []
    for single in (False, True):
        gb, fv = gpu_objects(g_io, cfg)
        prim = to_dev(gb.to_grid_order(ref))
        cons = torch.zeros((fv.ncons, gb.Nt), dtype=torch.float64, device="cuda")
        fv.prim_to_cons(prim, cons)
        w, d = prim.clone(), torch.zeros_like(cons)
        fv.compute_dudt(w, gb, d)
        dt0 = 0.5 * fv.estimate_dt(w)
        print(f"rk {kind} {method} single={single}", flush=True)
        a, b = butcher(method)
        s, t, dt_prev, dts = len(b), 0.0, 0.5 * dt0, []
        end = dt0 * 1.9
        rk = RungeKutta(fv, method, cfl=0.5, max_time=end, dt_init=0.5 * dt0)
        for _ in range(3):
            if not single:
                dts.append(rk.take_step(cons, prim))
                continue
            k = [torch.zeros_like(cons) for _ in range(s)]
            tmp, flow = torch.zeros_like(cons), torch.zeros_like(prim)

            def add(u0, u1, kj, c):
                check(lib().ibis_apply_time_derivative(fv._h, ptr(u0), ptr(u1), ptr(kj), float(c),
                                                       None), "apply")
            fv.compute_dudt(prim, gb, k[0])
            torch.cuda.synchronize()
            dt = min(0.5 * fv.estimate_dt(prim), 1.5 * dt_prev, end - t)
            for i in range(1, s):
                add(cons, tmp, k[0], a[i, 0] * dt)
                for j in range(1, i):
                    if a[i, j] >= 1e-14:
                        add(tmp, tmp, k[j], a[i, j] * dt)
                fv.cons_to_prim(tmp, flow)
                fv.compute_dudt(flow, gb, k[i])
            for i in range(s):
                add(cons, cons, k[i], b[i] * dt)
            fv.cons_to_prim(cons, prim)
            torch.cuda.synchronize()
            t, dt_prev = t + dt, dt
            dts.append(dt)
        torch.cuda.synchronize()
        out.append((dts, cons.cpu().numpy(), prim.cpu().numpy()))
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][2], out[1][2])


@pytest.mark.parametrize("mesh", ["wedge_2x1", "wedge_16x16", "wedge_17x16", "wedge_256x256",
                                  "wedge_257x256", "plate_37x19", "hex_9"])
def test_face_kernel_with_a_thread_per_face(mesh):
    """The blocks of the face kernel have a thread per face up to one tile per
    CU (256 tiles, 65,536 cells) and the tile's threads beyond: the residual's
    bits are those of 128- and 512-cell tiles, as each cell sums its faces in
    its own order."""
    import torch
    kind, size = mesh.split("_")
    if kind == "hex":
        g_io, cfg = cases.hex_case(int(size))
    else:
        nx, ny = map(int, size.split("x"))
        g_io, cfg = (cases.plate_case if kind == "plate" else cases.wedge_case)(nx, ny)[:2]
    out = []
    for tile in (256, 128, 512):
        gb, fv = gpu_objects(g_io, cfg)
        fv.set_option("tile", tile)
        prim = to_dev(gb.to_grid_order(
            cases.perturbed_prim(g_io, cases.freestream(2.0), gb.Nt, seed=31)))
        dudt = torch.zeros((fv.ncons, gb.Nt), dtype=torch.float64, device="cuda")
        fv.compute_dudt(prim, gb, dudt)
        out.append(dudt.cpu())
    assert torch.isfinite(out[0]).all()
    assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])


def _special_state(kind, grid_io, fs, nt):
    """States off the smooth path, from a uniform flow (3D: with a vz): noise
    in the last bit (every other cell is its own extremum, and most of the
    limiter's quotients tie at zero), a few plateaus (exact ties), a
    transverse velocity so small that products of two differences underflow,
    and single cells that are NaN, infinite, or so large that gradients
    overflow."""
    rng = np.random.default_rng(131)
    n = grid_io.num_cells
    prim = cases.uniform_prim(fs, n, nt)
    if grid_io.dim == 3:
        prim[6, :n] = 0.3 * fs.vx
    prim[:, n:] = prim[:, :1]
    if kind == "last_bit":
        prim[:, :n] += rng.integers(-1, 2, (7, n)) * np.spacing(prim[:, :n])
    elif kind == "plateaus":
        prim[:, :n] *= 1.0 + rng.integers(0, 3, (7, n)) / 64.0
    elif kind == "tiny":
        prim[5, :n] = rng.standard_normal(n) * 1e-302
    else:
        value = {"nan": np.nan, "inf": np.inf, "huge": 2e307}[kind]
        for k, row in enumerate((0, 3, 4, 5)):
            prim[row, n // 2 + 11 * k] = value if k != 3 else -value
    return prim


@pytest.mark.parametrize("kind", ["last_bit", "plateaus", "tiny", "nan", "inf", "huge"])
@pytest.mark.parametrize("limiter", ["barth_jespersen", "venkatakrishnan", "unlimited"])
@pytest.mark.parametrize("mesh", ["wedge", "triquad", "hex"])
def test_states_with_ties_and_non_finite_cells(mesh, limiter, kind):
    """The fused second-order path gives the oracle's bits (NaN in the same
    places) for the residual, the ghost rows, and the gradients and limiters
    it keeps. In 2D the z gradients, which it does not store, are left out."""
    import torch
    from ibis_amd import gridgen
    from ibis_amd.finite_volume import _device_view
    if mesh == "hex":
        g_io, cfg = cases.hex_case(9, flux="hanel", limiter=limiter)
        fs, nb = cases.freestream(2.0), 6 * 81
    else:
        g_io, cfg, fs = cases.wedge_case(32, 16, flux="hanel", limiter=limiter)
        g_io, nb = (gridgen.split_quads(g_io, 2) if mesh == "triquad" else g_io), 2 * (32 + 16)
    prim = _special_state(kind, g_io, fs, g_io.num_cells + nb)
    og, ofv = oracle_pair(g_io, cfg)
    p_cpu = prim.copy()
    with np.errstate(all="ignore"):
        d_cpu = ofv.compute_dudt(p_cpu)
    want = ofv.intermediates()
    n, dim = og.N, g_io.dim
    print(f"special state {kind} {mesh} {limiter} N={n}", flush=True)
    for opts in ({}, {"fold_boundary": 0}, {"stage_cells": 0}):
        gb, fv = gpu_objects(g_io, cfg)
        for k, v in opts.items():
            fv.set_option(k, v)
        fv.set_option("keep_gradients", 1)
        d_gpu, p_gpu = gpu_dudt(gb, fv, prim)
        g_ptr, l_ptr, _, _ = fv.scratch()
        grads = _device_view(g_ptr, (7, 3, n)).cpu().numpy()[..., gb.cell_new_of_old[:n]]
        lims = _device_view(l_ptr, (7, n)).cpu().numpy()[..., gb.cell_new_of_old[:n]]
        assert np.array_equal(d_gpu[:, :n], d_cpu[:, :n], equal_nan=True), opts
        assert np.array_equal(p_gpu[:, n:], p_cpu[:, n:], equal_nan=True), opts
        assert np.array_equal(grads[:, :dim], want["grads"][:, :dim], equal_nan=True), opts
        if limiter != "unlimited":
            assert np.array_equal(lims, want["lim"], equal_nan=True), opts
        fv.close()
        gb.close()


def _brick_mesh(gb, nx):
    """The arrays of a 2D quad grid with nx cells a row, its cells merged in
    pairs along the rows, every other row shifted by one, as bricks are laid:
    hexagons (6 faces) and, where a row ends in half a brick, quads."""
    from ibis_amd.batch import _concat_grids
    arr, N, G, F, _, _ = _concat_grids([gb])
    col, row = np.arange(N) % nx, np.arange(N) // nx
    brick = (col + row % 2) // 2
    new_of, cells = np.full(N + G, -1), {}
    for c in range(N):
        cells.setdefault((row[c], brick[c]), []).append(c)
    cells = list(cells.values())
    M = len(cells)
    for k, cs in enumerate(cells):
        new_of[cs] = k
    new_of[N:] = M + np.arange(G)
    left, right = new_of[arr["face_left"]], new_of[arr["face_right"]]
    keep = left != right
    face_of = np.cumsum(keep) - 1
    vol = np.concatenate([[arr["volume"][cs].sum() for cs in cells], arr["volume"][N:]])
    cen = np.concatenate([np.array([(arr["centroid"][:, cs] * arr["volume"][cs]).sum(axis=1) /
                                    arr["volume"][cs].sum() for cs in cells]).T,
                          arr["centroid"][:, N:]], axis=1)
    off, faces, signs, nbrs, lsq = [0], [], [], [], np.zeros((3, M))
    for k, cs in enumerate(cells):
        sxx = sxy = syy = 0.0
        for c in cs:
            for j in range(arr["cell_face_off"][c], arr["cell_face_off"][c + 1]):
                f = arr["cell_faces"][j]
                if not keep[f]:
                    continue
                n = new_of[arr["cell_neighbours"][j]]
                faces.append(face_of[f])
                signs.append(arr["cell_outsigns"][j])
                nbrs.append(n)
                dx, dy = cen[:2, n] - cen[:2, k]
                sxx, sxy, syy = sxx + dx * dx, sxy + dx * dy, syy + dy * dy
        off.append(len(faces))
        r11 = np.sqrt(sxx)
        r12 = 1.0 / r11 * sxy
        lsq[:, k] = r11, r12, np.sqrt(syy - r12 * r12)
    out = {"face_left": left[keep], "face_right": right[keep],
           "face_geom": arr["face_geom"][:, keep], "cell_face_off": np.array(off),
           "cell_faces": np.array(faces), "cell_outsigns": np.array(signs, np.int32),
           "cell_neighbours": np.array(nbrs), "centroid": cen, "volume": vol, "lsq": lsq,
           "tag_off": arr["tag_off"], "bfaces": face_of[arr["bfaces"]]}
    return {k: np.ascontiguousarray(v) for k, v in out.items()}, M, G, int(keep.sum())


@pytest.mark.parametrize("case", ["barth_jespersen", "venkatakrishnan", "unlimited", "viscous"])
def test_2d_cells_with_up_to_six_faces(case):
    """The kernels with the 2D stencil in LDS unroll over four faces; cells
    with more (a caller's own mesh) must take the others. Residual, tangent,
    matvec and adjoint of a mesh of bricks: with the default options the bits
    of the general path on pairs (its value), of the other implementations and
    of the reference-shaped viscous path; in FP32 those without the stencil in
    LDS."""
    import ctypes as C
    from types import SimpleNamespace

    import torch

    from ibis_amd.finite_volume import FiniteVolume, GridBlock
    from ibis_amd.native import MeshDescStruct, check, lib, ptr

    visc, nx, ny = case == "viscous", 37, 18
    if visc:
        g_io, cfg, fs = cases.plate_case(nx, ny)
    else:
        g_io, cfg, fs = cases.wedge_case(nx, ny, limiter=case)
    gb = GridBlock(g_io, cfg, reorder=False)
    arr, N, G, F = _brick_mesh(gb, nx)
    assert np.diff(arr["cell_face_off"]).max() == 6
    d = MeshDescStruct()
    d.dim, d.ntags = 2, len(arr["tag_off"]) - 1
    d.n_cells, d.n_ghost, d.n_faces = N, G, F
    for k, v in arr.items():
        setattr(d, k, ptr(v))
    m = C.c_void_p()
    check(lib().ibis_mesh_create(C.byref(d), C.byref(m)), "ibis_mesh_create")
    fvs = []

    def make(**opts):
        fv = FiniteVolume(SimpleNamespace(_mesh=m, dim=2, Nt=N + G), cfg)
        fvs.append(fv)
        for k, v in opts.items():
            fv.set_option(k, v)
        return fv

    rng = np.random.default_rng(171)
    x, y = arr["centroid"][0, :N], arr["centroid"][1, :N]
    ref = cases.uniform_prim(fs, N, N + G)
    ref[:, N:] = ref[:, :1]
    wave = [np.sin(9.0 * x + 1.7 * k) * np.cos(11.0 * y - k) for k in range(3)]
    ref[0, :N] *= 1.0 + 0.05 * wave[0]
    ref[2, :N] *= 1.0 + 0.05 * wave[1]
    ref[1, :N], ref[3, :N] = ref[0, :N] * cfg.gas.R * ref[2, :N], cfg.gas.Cv * ref[2, :N]
    ref[5, :N] += 0.05 * fs.vx * wave[2]
    dot, bar = rng.standard_normal(ref.shape), rng.standard_normal((4, N + G))

    def zeros(rows):
        return torch.zeros((rows, N + G), dtype=torch.float64, device="cuda")

    def residual(fv):
        p, out = to_dev(ref), zeros(4)
        fv.compute_dudt(p, None, out)
        torch.cuda.synchronize()
        return out.cpu().numpy()[:, :N], p.cpu().numpy()

    def tangent(fv):
        p, pd, out, od = to_dev(ref), to_dev(dot), zeros(4), zeros(4)
        fv.compute_dudt_jvp(p, pd, out, od)
        torch.cuda.synchronize()
        return [t.cpu().numpy() for t in (out[:, :N], p, od[:, :N], pd)]

    def reverse(fv, mode):
        p, pb = to_dev(ref), zeros(7)
        fv.compute_dudt_vjp(p, pb, dudt_bar=to_dev(bar), force_tags=7, force_dir=(0.3, 1.0, 0.0),
                            limiter=mode)
        torch.cuda.synchronize()
        return pb.cpu().numpy()

    try:
        print(f"bricks {case}: N={N} F={F}", flush=True)
        general = tangent(make(fuse_tangent=0))
        assert np.isfinite(general[0]).all() and np.abs(general[0]).max() > 0
        for a, b in zip(general, tangent(make())):
            assert np.array_equal(a, b)
        if visc:
            forms = [{}, {"fuse_viscous": 0}, {"fold_boundary": 0}]
        else:
            forms = [{}, {"fold_boundary": 0}, {"stage_cells": 0, "face_kernel": 128},
                     {"stage_cells": 0, "cell_prefetch": 1, "face_kernel": 0},
                     {"face_state_layout": 0, "face_kernel": 0, "precomputed_offsets": 0,
                      "stage_cells": 0, "pack_cells": 1}]
        out = [residual(make(**f)) for f in forms]
        for f, o in zip(forms, out):
            assert np.array_equal(o[0], out[-1][0]) and np.array_equal(o[1], general[1]), f
            if not visc:
                assert np.array_equal(o[0], general[0]), f
        for mode in ("fp32_flux", "fp32_recon") if not visc else ("fp32_flux",):
            a, b = make(), make(stage_cells=0) if not visc else make()
            a.set_precision(mode)
            b.set_precision(mode)
            f32 = residual(a)[0]
            assert np.array_equal(f32, residual(b)[0])
            assert (np.abs(f32 - out[0][0]).max(axis=1) < 1e-3 * np.abs(out[0][0]).max(axis=1)).all()
        for mode in ("active", "frozen"):
            want = reverse(make(vjp_tiles=0), mode)
            assert np.isfinite(want).all() and np.abs(want).max() > 0
            assert np.array_equal(reverse(make(), mode), want)
    finally:
        for fv in fvs:
            fv.close()
        lib().ibis_mesh_destroy(m)
        gb.close()
