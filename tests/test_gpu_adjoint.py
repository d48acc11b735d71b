"""The hand-written discrete adjoint of the residual.

Checks (as the reference has no adjoint, these are the definition of
correct):
  - dot-product test <w, J v> = <J^T w, v> with J v from the Dual tangent
    residual (itself equal to the oracle's FiniteVolume<Dual> bit for bit),
    relative to sum |w_i (J v)_i|, tolerance 1e-10; limiter active, and
    frozen against the tangent residual with the limiter frozen;
  - the gradient of the wall force functional against central finite
    differences of the force (step 1e-7 relative to the state, 32 seeded
    directions, seed 6);
  - the torch.autograd.Function wrappers return the same bars.
"""
import numpy as np
import pytest

from helpers import gpu_objects, to_dev
from ibis_amd import cases

pytestmark = pytest.mark.gpu

TOL = 1e-10


def _scale(prim, n):
    return np.abs(prim[:, :n]).max(axis=1) * 1e-3 + 1e-6


def _dot(g_io, cfg, prim_ref, seed, limiter="active"):
    import torch
    gb, fv = gpu_objects(g_io, cfg)
    N, Nt, nc = gb.N, gb.Nt, gb.dim + 2
    prim0 = gb.to_grid_order(prim_ref)
    rng = np.random.default_rng(seed)
    v = rng.standard_normal((7, Nt)) * _scale(prim0, N)[:, None]
    w = rng.standard_normal((nc, Nt))
    w[:, N:] = 0.0
    fv.set_option("freeze_limiter", 1 if limiter == "frozen" else 0)
    dudt = torch.zeros((nc, Nt), dtype=torch.float64, device="cuda")
    ddot = torch.zeros_like(dudt)
    fv.compute_dudt_jvp(to_dev(prim0), to_dev(v), dudt, ddot)
    pb = torch.zeros((7, Nt), dtype=torch.float64, device="cuda")
    fv.compute_dudt_vjp(to_dev(prim0), pb, dudt_bar=to_dev(w), limiter=limiter)
    torch.cuda.synchronize()
    jv = ddot.cpu().numpy()[:, :N]
    pbh = pb.cpu().numpy()
    lhs = float((w[:, :N] * jv).sum())
    rhs = float((pbh[:, :N] * v[:, :N]).sum())
    mag = float(np.abs(w[:, :N] * jv).sum())
    assert np.all(pbh[:, N:] == 0.0)
    assert mag > 0.0
    rel = abs(lhs - rhs) / mag
    print(f"dot test N={N} flux={cfg.flux} lim={cfg.limiter} visc={cfg.viscous} "
          f"mode={limiter}: <w,Jv>={lhs:.15e} <JTw,v>={rhs:.15e} rel={rel:.2e}", flush=True)
    assert rel < TOL
    return gb, fv


@pytest.mark.parametrize("flux,limiter", [("ausmdv", "barth_jespersen"), ("hanel", "venkatakrishnan"),
                                          ("rusanov", "unlimited")])
@pytest.mark.parametrize("mode", ["active", "frozen"])
def test_dot_product_wedge(flux, limiter, mode):
    g_io, cfg, fs = cases.wedge_case(48, 24, flux=flux, limiter=limiter)
    prim = cases.perturbed_prim(g_io, fs, 48 * 24 + 2 * (48 + 24), seed=81)
    _dot(g_io, cfg, prim, seed=82, limiter=mode)


@pytest.mark.parametrize("mode", ["active", "frozen"])
def test_dot_product_plate_viscous(mode):
    g_io, cfg, fs = cases.plate_case(64, 32)
    prim = cases.perturbed_prim(g_io, fs, 64 * 32 + 2 * (64 + 32), seed=2)
    _dot(g_io, cfg, prim, seed=83, limiter=mode)


def test_dot_product_hex():
    g_io, cfg = cases.hex_case(10, flux="hanel", limiter="venkatakrishnan")
    prim = cases.hex_prim(g_io, 10 ** 3 + 6 * 10 ** 2)
    _dot(g_io, cfg, prim, seed=84, limiter="active")


def test_dot_product_mixed_hex_pyramid():
    from ibis_amd import gridgen
    g_io, cfg = cases.hex_case(8, flux="hanel", limiter="venkatakrishnan")
    gh = gridgen.split_hexes(g_io, 3)
    prim = cases.hex_prim(gh, gh.num_cells + 6 * 64)
    _dot(gh, cfg, prim, seed=85, limiter="active")


@pytest.mark.parametrize("case", ["wedge_ausmdv", "wedge_hanel", "plate_viscous"])
def test_dot_product_first_order(case):
    """First-order residual (copy_reconstruct, convective_flux.cpp:212-240):
    the face states are the cells' whole prim rows."""
    if case == "plate_viscous":
        g_io, cfg, fs = cases.plate_case(48, 24)
        cfg.reconstruction_order = 1
        prim = cases.perturbed_prim(g_io, fs, 48 * 24 + 2 * (48 + 24), seed=86)
    else:
        g_io, cfg, fs = cases.wedge_case(48, 24, flux=case.split("_")[1], order=1)
        prim = cases.perturbed_prim(g_io, fs, 48 * 24 + 2 * (48 + 24), seed=87)
    _dot(g_io, cfg, prim, seed=88, limiter="frozen")


@pytest.mark.parametrize("order,mode", [(2, "active"), (2, "frozen"), (1, "frozen")])
def test_dot_product_subsonic_boundaries(order, mode):
    """Subsonic inflow and outflow ghosts (boundary.cpp:286-399) backwards,
    with a slip wall, on a Mach 0.5 wedge."""
    from ibis_amd import config as C
    g_io, cfg, fs = cases.wedge_case(48, 24, mach=0.5, order=order)
    cfg.boundaries = {"inflow": C.subsonic_inflow(fs), "outflow": C.subsonic_outflow(fs.p * 0.98),
                      "wall": C.slip_wall()}
    prim = cases.perturbed_prim(g_io, fs, 48 * 24 + 2 * (48 + 24), seed=89)
    _dot(g_io, cfg, prim, seed=90, limiter=mode)


@pytest.mark.parametrize("viscous", [False, True])
def test_dot_product_constant_flux_boundary(viscous):
    """A constant-flux inflow (boundary.cpp:405-443): its faces' convective
    flux is a constant; the viscous flux on them still depends on the state."""
    from ibis_amd import config as C
    g_io, cfg, fs = cases.wedge_case(48, 24, mach=2.0)
    cfg.boundaries = {"inflow": C.constant_flux(fs), "outflow": C.supersonic_outflow(),
                      "wall": C.fixed_temperature_no_slip_wall(300.0) if viscous else C.slip_wall()}
    cfg.viscous = viscous
    prim = cases.perturbed_prim(g_io, fs, 48 * 24 + 2 * (48 + 24), seed=91)
    _dot(g_io, cfg, prim, seed=92, limiter="active")


def test_wall_force_gradient_central_differences():
    """Config-4 check on a 64 x 32 flat plate: d J / d prim . v against
    (J(p + h v) - J(p - h v)) / 2h, h = 1e-7, 32 directions (seed 6)."""
    import torch
    g_io, cfg, fs = cases.plate_case(64, 32)
    prim_ref = cases.perturbed_prim(g_io, fs, 64 * 32 + 2 * (64 + 32), seed=2)
    gb, fv = gpu_objects(g_io, cfg)
    N, Nt = gb.N, gb.Nt
    prim0 = gb.to_grid_order(prim_ref)
    tags = fv.tag_mask("wall")
    for direction in ((1.0, 0.0, 0.0), (0.0, 1.0, 0.0)):
        pb = torch.zeros((7, Nt), dtype=torch.float64, device="cuda")
        fv.compute_dudt_vjp(to_dev(prim0), pb, force_tags=tags, force_dir=direction)
        grad = pb.cpu().numpy()
        rng = np.random.default_rng(6)
        errs = []
        h = 1e-7
        for k in range(32):
            v = rng.standard_normal((7, Nt)) * np.abs(prim0[:, :N]).max(axis=1)[:, None]
            v[:, N:] = 0.0
            # rho_u state: keep p, T, e consistent is not needed, the
            # residual reads rho, e, v (and T, v in the viscous flux)
            fp = fv.wall_force(to_dev(prim0 + h * v), tags) @ np.array(direction)
            fm = fv.wall_force(to_dev(prim0 - h * v), tags) @ np.array(direction)
            fd = (fp - fm) / (2 * h)
            ad = float((grad[:, :N] * v[:, :N]).sum())
            errs.append(abs(fd - ad) / max(abs(ad), 1e-300))
        errs = np.array(errs)
        print(f"force dir {direction}: FD rel err median {np.median(errs):.2e} max {errs.max():.2e}",
              flush=True)
        assert np.median(errs) < 1e-6
        assert errs.max() < 1e-4


def test_autograd_functions_match_vjp():
    import torch
    from ibis_amd.autograd import residual, wall_force
    g_io, cfg, fs = cases.plate_case(32, 16)
    prim_ref = cases.perturbed_prim(g_io, fs, 32 * 16 + 2 * (32 + 16), seed=2)
    gb, fv = gpu_objects(g_io, cfg)
    N, Nt = gb.N, gb.Nt
    prim0 = to_dev(gb.to_grid_order(prim_ref))
    x = prim0.clone().requires_grad_(True)
    J = wall_force(x, fv, "wall", (1.0, 0.0, 0.0))
    J.backward()
    pb = torch.zeros_like(prim0)
    fv.compute_dudt_vjp(prim0.clone(), pb, force_tags=fv.tag_mask("wall"))
    assert torch.equal(x.grad, pb)
    assert float(J.detach()) == float(fv.wall_force(prim0.clone(), fv.tag_mask("wall"))[0])
    y = prim0.clone().requires_grad_(True)
    d = residual(y, fv)
    w = torch.randn(d.shape, dtype=torch.float64, device="cuda", generator=torch.Generator(
        device="cuda").manual_seed(7))
    w[:, N:] = 0.0
    (d * w).sum().backward()
    pb2 = torch.zeros_like(prim0)
    fv.compute_dudt_vjp(prim0.clone(), pb2, dudt_bar=w.contiguous())
    assert torch.equal(y.grad, pb2)


def _reverse_forms():
    C, G = cases.C, cases.gridgen
    fs = cases.freestream(0.5)
    sub = C.FVConfig(flux="hanel", boundaries={
        "inflow": C.subsonic_inflow(fs), "outflow": C.subsonic_outflow(101325.0),
        "wall": C.adiabatic_no_slip_wall()})
    wedge = lambda nx=37, ny=19, **kw: cases.wedge_case(nx, ny, **kw)[:2]  # noqa: E731
    const = wedge()
    const[1].boundaries["inflow"] = C.constant_flux(cases.freestream(3.0))
    walled = cases.hex_case(7, flux="ausmdv", limiter="barth_jespersen")
    walled[1].viscous = True
    walled[1].boundaries["bottom"] = C.fixed_temperature_no_slip_wall(320.0)
    return {
        "wedge": wedge(), "one_tile": wedge(16, 8), "one_over": wedge(43, 3), "one_under": wedge(127, 1),
        "hanel_venkat_rho_p": wedge(flux="hanel", limiter="venkatakrishnan", thermo="rho_p"),
        "rusanov_unlimited_pT": wedge(flux="rusanov", limiter="unlimited", thermo="p_T"),
        "rho_T": wedge(thermo="rho_T"), "subsonic": (G.wedge(24, 12), sub), "constant_flux": const,
        "plate": cases.plate_case(33, 17)[:2], "hex": cases.hex_case(9), "hex_viscous": walled,
        "triangles": (G.split_quads(G.wedge(20, 10)), wedge()[1]),
        "pyramids": (G.split_hexes(G.hex_box(6)), cases.hex_case(4)[1]),
    }


@pytest.mark.parametrize("name", sorted(_reverse_forms()))
@pytest.mark.parametrize("limiter", ["active", "frozen"])
def test_tile_reverse_equals_face_and_cell_kernels(name, limiter):
    """The reverse by tiles gives the bits of the kernels over face-indexed
    arrays: each face's and cell's expressions and the order of every sum are
    the same, and a border face is evaluated by both its tiles alike."""
    import torch
    g_io, cfg = _reverse_forms()[name]
    rng = np.random.default_rng(83)
    out = []
    for tiles in (0, 1):
        gb, fv = gpu_objects(g_io, cfg)
        fv.set_option("vjp_tiles", tiles)
        if tiles == 0:
            ref = cases.perturbed_prim(g_io, cases.freestream(2.0), gb.Nt, seed=84)
            ref[6, :gb.N] = 20.0 * np.sin(np.arange(gb.N))
            w = rng.standard_normal((fv.ncons, gb.Nt))
        prim = to_dev(gb.to_grid_order(ref))
        bar = torch.full_like(prim, float("nan"))
        print(f"reverse {name} {limiter} tiles={tiles}", flush=True)
        fv.compute_dudt_vjp(prim, bar, dudt_bar=to_dev(gb.to_grid_order(w)),
                            force_tags=(1 << len(gb.tags)) - 1, force_dir=(0.3, 1.0, -0.7),
                            limiter=limiter)
        torch.cuda.synchronize()
        out.append((bar.cpu().numpy(), prim.cpu().numpy()))
    assert np.isfinite(out[0][0]).all() and np.abs(out[0][0]).max() > 0
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


def _force_forms():
    wedge = lambda nx, ny, **kw: cases.wedge_case(nx, ny, **kw)[:2]  # noqa: E731
    hexes = lambda n, **kw: cases.hex_case(n, **kw)  # noqa: E731
    return {
        "few_faces": wedge(2, 1), "one_wave": wedge(21, 11), "one_over": wedge(32, 33),
        "venkat_rho_p": wedge(37, 19, flux="hanel", limiter="venkatakrishnan", thermo="rho_p"),
        "unlimited_pT": wedge(37, 19, flux="rusanov", limiter="unlimited", thermo="p_T"),
        "rho_T": wedge(37, 19, thermo="rho_T"), "ldfss2": wedge(37, 19, flux="ldfss2"),
        "hex": hexes(9), "hex_bj": hexes(5, flux="ausmdv", limiter="barth_jespersen"),
    }


@pytest.mark.parametrize("name", sorted(_force_forms()))
def test_wall_force_balances_the_momentum(name):
    """The inner faces' fluxes cancel in sum_c V_c dU_c/dt, so the force on
    all boundaries is minus that sum of the momentum rows; and the boundaries'
    own forces add up to it.  Rounding: no flux * area exceeds the largest
    area times twice the largest p + rho |v|^2 of the state, each of the F
    faces enters at most twice, and no partial sum has more than F roundings
    and the few of its terms: (F + 8) eps of that total."""
    import torch
    g_io, cfg = _force_forms()[name]
    gb, fv = gpu_objects(g_io, cfg)
    N = gb.N
    prim = gb.to_grid_order(cases.perturbed_prim(g_io, cases.freestream(2.0), gb.Nt, seed=97))
    dudt = torch.zeros((fv.ncons, gb.Nt), dtype=torch.float64, device="cuda")
    fv.compute_dudt(to_dev(prim), gb, dudt)
    geo = gb.export()
    terms = dudt.cpu().numpy()[1:1 + gb.dim, :N] * geo["volume"][:N]
    x = to_dev(prim)
    force = fv.wall_force(x, (1 << len(gb.tags)) - 1)
    again = fv.wall_force(to_dev(prim), (1 << len(gb.tags)) - 1)
    single = [fv.wall_force(to_dev(prim), 1 << t) for t in range(len(gb.tags))]
    y = to_dev(prim)
    fv.compute_dudt(y, gb, dudt)
    assert torch.equal(x, y)  # the ghosts too
    assert np.array_equal(force, again)
    xh = x.cpu().numpy()
    top = (xh[1] + xh[0] * (xh[4:] ** 2).sum(axis=0)).max()
    tol = 2.0 ** -52 * (gb.F + 8) * 2 * gb.F * 2 * top * geo["face_geom"][12].max()
    print(f"force {name}: {force} sum {terms.sum(axis=1)} tol {tol:.1e}", flush=True)
    assert np.abs(force[:gb.dim] + terms.sum(axis=1)).max() <= tol
    assert np.abs(np.sum(single, axis=0) - force).max() <= tol
    assert np.all(force[gb.dim:] == 0.0) and np.array_equal(fv.wall_force(x, 0), np.zeros(3))


@pytest.mark.parametrize("kind", ["smooth", "plateaus", "nan", "inf"])
@pytest.mark.parametrize("name", sorted(_force_forms()) + ["triangles", "pyramids", "subsonic"])
def test_wall_force_from_the_boundary_equals_the_residuals_fluxes(name, kind):
    """An inviscid second-order residual's force is formed from its boundary's
    cells and faces alone, and has the bits of the sum over the general path's
    face fluxes. That path still serves residuals with a constant-flux
    boundary: with one tag made such (its ghosts as before), the other tags'
    forces must not change, NaN in the same places."""
    import copy

    from test_gpu_residual import _special_state
    C = cases.C
    form = {**_force_forms(), **{k: _reverse_forms()[k] for k in ("triangles", "pyramids", "subsonic")}}
    g_io, cfg = form[name]
    fs = cases.freestream(2.0)
    tags = sorted(cfg.boundaries)
    gb, fv = gpu_objects(g_io, cfg)
    if kind == "smooth":
        ref = cases.perturbed_prim(g_io, fs, gb.Nt, seed=98)
    else:
        if gb.N < 64:
            pytest.skip("too few cells for the marked ones")
        ref = _special_state(kind, g_io, fs, gb.Nt)
    prim = to_dev(gb.to_grid_order(ref))
    want = {t: fv.wall_force(prim.clone(), fv.tag_mask([t])) for t in tags}
    print(f"force {name} {kind}: {want}", flush=True)
    for fixed in tags:
        c2 = copy.deepcopy(cfg)
        c2.boundaries[fixed].post_convective_flux = C.constant_flux(fs).post_convective_flux
        gb2, fv2 = gpu_objects(g_io, c2)
        for t in tags:
            if t != fixed:
                got = fv2.wall_force(prim.clone(), fv2.tag_mask([t]))
                assert np.array_equal(got, want[t], equal_nan=True), (fixed, t)
        fv2.close()
        gb2.close()
    fv.close()
    gb.close()
