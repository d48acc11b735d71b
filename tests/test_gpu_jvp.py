"""Parity of the tangent (JVP) residual with the oracle's Dual residual.

ibis_compute_dudt_jvp replaces FiniteVolume<Ibis::dual> under
SteadyStateLinearisation::matrix_vector_product
(src/solvers/solvers/steady_state.cpp:52-128).  Inviscid cases compare both
the value and the tangent bit for bit (same Dual expression trees,
contraction disabled on both sides); cases that go through pow() (viscous
Sutherland, LDFSS2) compare at 1e-12 relative per conserved variable.
"""
import numpy as np
import pytest

from helpers import gpu_objects, oracle_pair, rel_err, to_dev
from ibis_amd import cases

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _tangent(shape, seed, scale):
    rng = np.random.default_rng(seed)
    return rng.standard_normal(shape) * scale[:, None]


def _jvp_case(grid_io, cfg, prim_ref, seed, exact, allow_reconstruction=True, nan_ok=False):
    import torch
    og, ofv = oracle_pair(grid_io, cfg)
    n, nt = og.N, og.N + og.G
    scale = np.abs(prim_ref[:, :n]).max(axis=1) * 1e-3 + 1e-3
    pdot_ref = _tangent(prim_ref.shape, seed, scale)
    p_cpu, pd_cpu = prim_ref.copy(), pdot_ref.copy()
    d_cpu, dd_cpu = ofv.compute_dudt_jvp(p_cpu, pd_cpu, allow_reconstruction)
    gb, fv = gpu_objects(grid_io, cfg)
    prim = to_dev(gb.to_grid_order(prim_ref))
    pdot = to_dev(gb.to_grid_order(pdot_ref))
    dudt = torch.zeros((gb.dim + 2, nt), dtype=torch.float64, device="cuda")
    ddot = torch.zeros_like(dudt)
    print(f"jvp case N={n} flux={cfg.flux} lim={cfg.limiter} visc={cfg.viscous} "
          f"recon={allow_reconstruction}", flush=True)
    fv.compute_dudt_jvp(prim, pdot, dudt, ddot, allow_reconstruction)
    torch.cuda.synchronize()
    d_gpu = gb.to_reference_order(dudt.cpu().numpy())
    dd_gpu = gb.to_reference_order(ddot.cpu().numpy())
    p_gpu = gb.to_reference_order(prim.cpu().numpy())
    pd_gpu = gb.to_reference_order(pdot.cpu().numpy())
    if nan_ok:
        # NaN tangents where the oracle has them (same positions), the rest
        # compared like any other tangent
        bad = ~np.isfinite(dd_cpu[:, :n])
        assert np.array_equal(bad, ~np.isfinite(dd_gpu[:, :n]))
        dd_cpu, dd_gpu = np.where(np.isfinite(dd_cpu), dd_cpu, 0.0), np.where(
            np.isfinite(dd_gpu), dd_gpu, 0.0)
    assert np.isfinite(dd_cpu[:, :n]).all() and np.abs(dd_cpu[:, :n]).max() > 0
    if exact:
        assert np.array_equal(d_gpu[:, :n], d_cpu[:, :n]), rel_err(d_gpu, d_cpu, n)
        assert np.array_equal(dd_gpu[:, :n], dd_cpu[:, :n]), rel_err(dd_gpu, dd_cpu, n)
    else:
        assert (rel_err(d_gpu, d_cpu, n) <= TOL).all(), rel_err(d_gpu, d_cpu, n)
        assert (rel_err(dd_gpu, dd_cpu, n) <= TOL).all(), rel_err(dd_gpu, dd_cpu, n)
    # ghost rows of the value and the tangent written by the boundary actions
    assert np.array_equal(p_gpu[:, n:], p_cpu[:, n:])
    assert np.array_equal(pd_gpu[:, n:], pd_cpu[:, n:])
    # the value part is the plain residual
    d_plain = ofv.compute_dudt(prim_ref.copy(), allow_reconstruction=allow_reconstruction)
    if exact:
        assert np.array_equal(d_gpu[:, :n], d_plain[:, :n])
    return og, ofv, gb, fv


@pytest.mark.parametrize("kw", [
    dict(flux="ausmdv", limiter="barth_jespersen", thermo="rho_u"),
    dict(flux="hanel", limiter="venkatakrishnan", thermo="rho_p"),
    dict(flux="rusanov", limiter="unlimited", thermo="p_T"),
], ids=lambda k: "-".join(k.values()))
def test_wedge_jvp(kw):
    g_io, cfg, fs = cases.wedge_case(48, 24, **kw)
    prim = cases.perturbed_prim(g_io, fs, 48 * 24 + 2 * (48 + 24), seed=31)
    _jvp_case(g_io, cfg, prim, seed=32, exact=True)


def test_wedge_jvp_first_order_preconditioner():
    """allow_reconstruction = false, as the JFNK preconditioner runs it
    (steady_state.cpp:47-50)."""
    g_io, cfg, fs = cases.wedge_case(48, 24)
    prim = cases.perturbed_prim(g_io, fs, 48 * 24 + 2 * (48 + 24), seed=33)
    _jvp_case(g_io, cfg, prim, seed=34, exact=True, allow_reconstruction=False)


def test_wedge_jvp_ldfss2():
    """The reference's Dual pow (UT/dual.h:239-245) adds power.dual *
    real * log(base): with a constant exponent that is 0 * log(base), NaN
    for the negative base LDFSS2 passes it on subsonic faces
    (ldfss2.cpp, (sqrt(0.5 (ML^2 + MR^2)) - 1)^2).  The tangent is NaN there
    in the reference, the oracle and here alike."""
    g_io, cfg, fs = cases.wedge_case(48, 24, flux="ldfss2")
    prim = cases.perturbed_prim(g_io, fs, 48 * 24 + 2 * (48 + 24), seed=35)
    _jvp_case(g_io, cfg, prim, seed=36, exact=False, nan_ok=True)


def test_hex_jvp():
    g_io, cfg = cases.hex_case(12, flux="hanel", limiter="venkatakrishnan")
    prim = cases.hex_prim(g_io, 12 ** 3 + 6 * 12 ** 2)
    _jvp_case(g_io, cfg, prim, seed=37, exact=True)


def test_mixed_elements_jvp():
    """Tangent residual on ragged stencils: triangle / quad and hex / pyramid."""
    from ibis_amd import gridgen
    g_io, cfg, fs = cases.wedge_case(24, 12)
    gm = gridgen.split_quads(g_io, 2)
    prim = cases.perturbed_prim(gm, fs, gm.num_cells + 2 * (24 + 12), seed=33)
    _jvp_case(gm, cfg, prim, seed=38, exact=True)
    g_io, cfg = cases.hex_case(8, flux="hanel", limiter="venkatakrishnan")
    gh = gridgen.split_hexes(g_io, 3)
    _jvp_case(gh, cfg, cases.hex_prim(gh, gh.num_cells + 6 * 64), seed=39, exact=True)


def test_plate_viscous_jvp():
    g_io, cfg, fs = cases.plate_case(64, 32)
    prim = cases.perturbed_prim(g_io, fs, 64 * 32 + 2 * (64 + 32), seed=2)
    _jvp_case(g_io, cfg, prim, seed=38, exact=False)


def test_cons_to_prim_jvp():
    import torch
    g_io, cfg, fs = cases.wedge_case(48, 24)
    nt = 48 * 24 + 2 * (48 + 24)
    prim = cases.perturbed_prim(g_io, fs, nt, seed=39)
    og, ofv = oracle_pair(g_io, cfg)
    cons = ofv.prim_to_cons(prim)
    cdot = np.random.default_rng(40).standard_normal(cons.shape)
    p_cpu, pd_cpu = ofv.cons_to_prim_jvp(cons, cdot)
    gb, fv = gpu_objects(g_io, cfg)
    p = torch.zeros((7, nt), dtype=torch.float64, device="cuda")
    pd = torch.zeros_like(p)
    fv.cons_to_prim_jvp(to_dev(gb.to_grid_order(cons)), to_dev(gb.to_grid_order(cdot)), p, pd)
    torch.cuda.synchronize()
    n = og.N
    assert np.array_equal(gb.to_reference_order(p.cpu().numpy())[:, :n], p_cpu[:, :n])
    assert np.array_equal(gb.to_reference_order(pd.cpu().numpy())[:, :n], pd_cpu[:, :n])


def _tangent_forms():
    fs = cases.freestream(0.5)
    sub = cases.C.FVConfig(flux="ausmdv", boundaries={
        "inflow": cases.C.subsonic_inflow(fs), "outflow": cases.C.subsonic_outflow(101325.0),
        "wall": cases.C.adiabatic_no_slip_wall()})
    plate = lambda **kw: cases.plate_case(33, 17, **kw)[:2]  # noqa: E731
    wedge = lambda nx=37, ny=19, **kw: cases.wedge_case(nx, ny, **kw)[:2]  # noqa: E731
    walled = cases.hex_case(7, flux="ausmdv", limiter="barth_jespersen")
    walled[1].viscous = True
    walled[1].boundaries["bottom"] = cases.C.fixed_temperature_no_slip_wall(320.0)
    tri = cases.gridgen.split_quads(cases.gridgen.wedge(20, 10))
    pyr = cases.gridgen.split_hexes(cases.gridgen.hex_box(6))
    return {
        "wedge": wedge(), "wedge_one_tile": wedge(16, 16), "wedge_tail": wedge(257, 1),
        "hanel_venkat_rho_p": wedge(flux="hanel", limiter="venkatakrishnan", thermo="rho_p"),
        "rusanov_unlimited_pT": wedge(flux="rusanov", limiter="unlimited", thermo="p_T"),
        "ldfss2": wedge(flux="ldfss2", thermo="rho_T"), "order1": wedge(order=1),
        "subsonic": (cases.gridgen.wedge(24, 12), sub),
        "plate": plate(), "plate_hanel": plate(flux="hanel"), "hex": cases.hex_case(9),
        "hex_viscous": walled, "triangles": (tri, wedge()[1]), "pyramids": (pyr, cases.hex_case(4)[1]),
    }


@pytest.mark.parametrize("name", sorted(_tangent_forms()))
@pytest.mark.parametrize("tile", [128, 256])
def test_fused_tangent_equals_general_path(name, tile):
    """The three- or four-kernel tangent residual and steady matvec give the
    general path's bits (NaN in the same places) for values, tangents, ghost
    rows and matvec results: with and without reconstruction, with a frozen
    limiter, twice in a row (the 2D vz gradient of a call is the viscous one
    of the call before, so the states have a vz)."""
    import torch
    from ibis_amd.steady import SteadyStateLinearisation
    g_io, cfg = _tangent_forms()[name]
    rng = np.random.default_rng(77)
    res = {}
    for fused in (0, 1):
        gb, fv = gpu_objects(g_io, cfg)
        fv.set_option("tile", tile)
        fv.set_option("fuse_tangent", fused)
        if fused == 0:
            fs = cases.freestream(2.0)
            ref = cases.perturbed_prim(g_io, fs, gb.Nt, seed=78)
            ref[6, :gb.N] = 0.1 * fs.vx * np.sin(np.arange(gb.N))
            ref[:, gb.N:] = ref[:, :1]
            dot = rng.standard_normal(ref.shape) * 1e-3 * np.abs(ref).max(axis=1)[:, None]
            vec = rng.standard_normal(gb.N * fv.ncons)
        out = []
        for freeze in (0, 1):
            fv.set_option("freeze_limiter", freeze)
            for recon in (True, False, True):
                prim = to_dev(gb.to_grid_order(ref))
                pdot = to_dev(gb.to_grid_order(dot))
                dudt = torch.zeros((fv.ncons, gb.Nt), dtype=torch.float64, device="cuda")
                ddot = torch.zeros_like(dudt)
                print(f"tangent {name} tile={tile} fused={fused} freeze={freeze} recon={recon}",
                      flush=True)
                fv.compute_dudt_jvp(prim, pdot, dudt, ddot, recon)
                cons = torch.zeros_like(dudt)
                fv.prim_to_cons(prim, cons)
                op = SteadyStateLinearisation(fv, cons, recon)
                op.set_pseudo_time_step(3e-6)
                w = torch.zeros(gb.N * fv.ncons, dtype=torch.float64, device="cuda")
                op.matrix_vector_product(to_dev(vec), w)
                torch.cuda.synchronize()
                out += [t.cpu().numpy() for t in (dudt, ddot, prim, pdot, w)]
        res[fused] = out
    for a, b in zip(res[0], res[1]):
        assert np.array_equal(a, b, equal_nan=True)
