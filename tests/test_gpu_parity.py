"""GPU parity of every hot-path function against the oracle and the reference's golden vectors.

Bit-exact: geometry, CSR structure and slot maps, Laplacian and
convection-diffusion assembly, face fluxes and divergence, SpMV, DIC/DILU
pivots and the triangular sweeps (all run the reference's per-row order).
Solvers: with the sums in index order (fc_set_reduction_order SEQUENTIAL)
the reference's solution, residual and iteration count bit for bit; with the
default tree-ordered sums the reference's iteration counts within one, and
after the reference's number of iterations its iterate within 1e-9 relative
FP64 residual.
"""
import numpy as np
import pytest

from conftest import (ADJUST_CASES, BC_CASES, CALCP_CASES, CALCP_FIELDS, CONVDIFF_CASES, GRAD_CASES, MESH_CASES,
                      PISO_FIELDS, calcp_uniform_case, load_transcript)
from freecappuccino_amd import fcap
from freecappuccino_amd import mesh as M
from freecappuccino_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = fcap.Context(0)
    yield c
    c.close()


def _csr_of(g):
    m = g.mesh
    return fcap.CSR(*(g.out(g.first, k) for k in ("ioffset", "ja", "diag", "ij_slot", "ji_slot")))


def _geo_of(g):
    return fcap.Geometry(*(g.out(g.first, k) for k in ("arx", "ary", "arz", "xf", "yf", "zf", "vol", "xc", "yc",
                                                       "zc", "facint")))


@pytest.mark.parametrize("case", MESH_CASES + CONVDIFF_CASES)
def test_geometry_bitwise(ctx, golden_loader, case):
    g = golden_loader(case)
    geo = fcap.mesh_geometry(g.mesh, ctx)
    for k in ("arx", "ary", "arz", "xf", "yf", "zf", "vol", "xc", "yc", "zc", "facint"):
        np.testing.assert_array_equal(getattr(geo, k), g.out(g.first, k), err_msg=k)


@pytest.mark.parametrize("case", MESH_CASES + CONVDIFF_CASES)
def test_csr_bitwise(ctx, golden_loader, case):
    g = golden_loader(case)
    m = g.mesh
    c = fcap.create_csr_matrix_from_mesh_data(m.n_cells, m.owner[:m.n_inner] + 1, m.neighbour + 1, ctx)
    for k in ("ioffset", "ja", "diag", "ij_slot", "ji_slot"):
        np.testing.assert_array_equal(getattr(c, k), g.out(g.first, k), err_msg=k)


@pytest.mark.parametrize("case", MESH_CASES)
def test_laplacian_bitwise(ctx, golden_loader, case):
    g = golden_loader(case)
    a, su = fcap.laplacian(g.mesh, _geo_of(g), _csr_of(g), g.inp("mu"), g.inp("phi"), g.inp("su0"), ctx)
    np.testing.assert_array_equal(a, g.out(g.first, "a"))
    np.testing.assert_array_equal(su, g.out(g.first, "su"))


def test_laplacian_wall_values_bitwise(ctx, golden_loader):
    """Non-zero Dirichlet values and a non-constant mu exercise su += a(diag)*phi_b (fvm_laplacian.f90:152)."""
    g = golden_loader("hex6x5x4_graded")
    m = g.mesh
    rng = np.random.default_rng(5)
    mu = -rng.uniform(0.5, 2.0, m.n_cells)
    phi = rng.standard_normal(m.n_cells + m.n_boundary)
    su0 = rng.standard_normal(m.n_cells)
    geo, csr = _geo_of(g), _csr_of(g)
    a, su = fcap.laplacian(m, geo, csr, mu, phi, su0, ctx)
    og = O.Geometry(*(getattr(geo, k) for k in ("arx", "ary", "arz", "xf", "yf", "zf", "vol", "xc", "yc", "zc",
                                                "facint")))
    oc = O.CSR(csr.ioffset, csr.ja, csr.diag, csr.ij_slot, csr.ji_slot)
    a_o, su_o = O.laplacian(m, og, oc, mu, phi, su0)
    np.testing.assert_array_equal(a, a_o)
    np.testing.assert_array_equal(su, su_o)


@pytest.mark.parametrize("case", CONVDIFF_CASES)
def test_convdiff_and_fluxes_bitwise(ctx, golden_loader, case):
    g = golden_loader(case)
    m = g.mesh
    geo, csr = _geo_of(g), _csr_of(g)
    flux = fcap.face_flux_central(m, geo, g.inp("u"), g.inp("v"), g.inp("w"), ctx)
    np.testing.assert_array_equal(flux, g.inp("flux"))
    a = fcap.convdiff(m, geo, csr, g.inp("vis"), flux, 0.7, ctx)
    np.testing.assert_array_equal(a, g.inp("a_convdiff"))
    su = fcap.rhs_divergence(m, flux, np.zeros(m.n_cells), ctx)
    np.testing.assert_array_equal(su, O.rhs_divergence(m, flux, np.zeros(m.n_cells)))


@pytest.mark.parametrize("case", MESH_CASES)
def test_spmv_pivots_sweeps_bitwise(ctx, golden_loader, case):
    g = golden_loader(case)
    csr = _csr_of(g)
    oc = O.CSR(csr.ioffset, csr.ja, csr.diag, csr.ij_slot, csr.ji_slot)
    a = g.out(g.first, "a")
    x = np.random.default_rng(0).standard_normal(csr.diag.shape[0])
    np.testing.assert_array_equal(fcap.spmv(csr, a, x, ctx), O.spmv(oc, a, x))
    d = fcap.dic_pivots(csr, a, ctx)
    np.testing.assert_array_equal(d, O.dic_pivots(oc, a))
    np.testing.assert_array_equal(fcap.lu_apply(csr, a, d, x, ctx), O.lu_apply(oc, a, d, x))


@pytest.mark.parametrize("case", MESH_CASES + CONVDIFF_CASES)
def test_sweeps_dependent_schedule_bitwise(ctx, golden_loader, case):
    """Every schedule of the pivots and sweeps -- one launch per level, one launch per sweep with
    each row waiting for the rows it reads, and the part-wise sweeps -- gives the oracle's DIC and
    DILU values bit for bit."""
    g = golden_loader(case)
    csr = _csr_of(g)
    oc = O.CSR(csr.ioffset, csr.ja, csr.diag, csr.ij_slot, csr.ji_slot)
    dilu = case in CONVDIFF_CASES
    a = g.inp("a_convdiff") if dilu else g.out(g.first, "a")
    d_ref = O.dilu_pivots(oc, a) if dilu else O.dic_pivots(oc, a)
    r = np.random.default_rng(2).standard_normal(csr.diag.shape[0])
    ref = O.lu_apply(oc, a, d_ref, r)
    try:
        for mode in (fcap.SWEEP_LEVELS, fcap.SWEEP_DEPENDENT, fcap.SWEEP_PARTS):
            ctx.set_sweep_mode(mode)
            d = fcap.dilu_pivots(csr, a, ctx) if dilu else fcap.dic_pivots(csr, a, ctx)
            np.testing.assert_array_equal(d, d_ref, err_msg=f"pivots, mode {mode}")
            np.testing.assert_array_equal(fcap.lu_apply(csr, a, d, r, ctx), ref, err_msg=f"sweeps, mode {mode}")
    finally:
        ctx.set_sweep_mode(fcap.SWEEP_DEFAULT)


@pytest.mark.parametrize("case", CONVDIFF_CASES)
def test_dilu_pivots_bitwise(ctx, golden_loader, case):
    g = golden_loader(case)
    csr = _csr_of(g)
    oc = O.CSR(csr.ioffset, csr.ja, csr.diag, csr.ij_slot, csr.ji_slot)
    a = g.inp("a_convdiff")
    d = fcap.dilu_pivots(csr, a, ctx)
    np.testing.assert_array_equal(d, O.dilu_pivots(oc, a))
    r = np.random.default_rng(1).standard_normal(csr.diag.shape[0])
    np.testing.assert_array_equal(fcap.lu_apply(csr, a, d, r, ctx), O.lu_apply(oc, a, d, r))


def _dense(csr, a):
    import scipy.sparse as sp
    n = csr.diag.shape[0]
    return sp.csr_matrix((a, csr.ja - 1, csr.ioffset - 1), shape=(n, n))


@pytest.mark.parametrize("case", MESH_CASES)
@pytest.mark.parametrize("solver", ["iccg", "dpcg", "bicgstab"])
def test_solvers_bitwise_with_sequential_sums(ctx, golden_loader, case, solver):
    """With every dot product and norm formed in index order (fc_set_reduction_order
    SEQUENTIAL), as the reference's sum(...) forms it, the GPU solvers repeat the reference's
    arithmetic exactly -- SpMV, pivots, sweeps and vector updates already have its rounding
    sequence -- so the solution, the final residual vector, res0 and the iteration count equal
    the reference's own (golden vectors from the reference compiled in place) bit for bit."""
    g = golden_loader(case)
    csr = _csr_of(g)
    a, su = g.out(g.first, "a"), g.out(g.first, "su")
    ctx.set_reduction_order(fcap.REDUCE_SEQUENTIAL)
    try:
        r = getattr(fcap, solver)(csr, a, su, g.inp("fi0"), sor=float(g.inp("sor")[0]),
                                  nsw=int(g.inp("nsw")[0]), ctx=ctx)
    finally:
        ctx.set_reduction_order(fcap.REDUCE_TREE)
    assert r.status == 0
    assert r.info["iters"] == int(g.out(solver, "iters")[0])
    assert r.info["res0"] == float(g.out(solver, "resor")[0])
    np.testing.assert_array_equal(r.fi, g.out(solver, "fi"))
    np.testing.assert_array_equal(r.res, g.out(solver, "res"))


@pytest.mark.parametrize("case", MESH_CASES)
@pytest.mark.parametrize("solver", ["iccg", "dpcg", "bicgstab"])
def test_solvers_match_reference(ctx, golden_loader, case, solver):
    """The default (tree-ordered, full-speed) sums against the reference's golden solve.
    1. With the reference's sor: converged, with the reference's iteration count within one
       (the partial sums are added in a fixed tree, not sequentially, so the stopping test may
       cross sor one iteration earlier or later).
    2. With nsw = the reference's iteration count: the reference's iterate within 1e-9 relative
       FP64 residual, ||A (x_gpu - x_ref)||_2 / ||su||_2 (measured: at most 2.8e-10, on the
       graded box with Jacobi-PCG; 1e-14..1e-11 elsewhere)."""
    g = golden_loader(case)
    csr = _csr_of(g)
    a, su = g.out(g.first, "a"), g.out(g.first, "su")
    fn = getattr(fcap, solver)
    r = fn(csr, a, su, g.inp("fi0"), sor=float(g.inp("sor")[0]), nsw=int(g.inp("nsw")[0]), ctx=ctx)
    ref_iters = int(g.out(solver, "iters")[0])
    assert r.status == 0
    assert abs(r.info["iters"] - ref_iters) <= 1, (r.info["iters"], ref_iters)
    A = _dense(csr, a)
    bn = np.linalg.norm(su)
    res_gpu = np.linalg.norm(su - A @ r.fi) / bn
    assert abs(r.info["rel_l2"] - res_gpu) <= 1e-12 + 1e-6 * res_gpu

    r2 = fn(csr, a, su, g.inp("fi0"), sor=1e-30, nsw=ref_iters, ctx=ctx)
    assert r2.status == fcap.FC_NOT_CONVERGED and r2.info["iters"] == ref_iters
    assert np.linalg.norm(A @ (r2.fi - g.out(solver, "fi"))) / bn <= 1e-9


@pytest.mark.parametrize("case", CONVDIFF_CASES)
def test_bicgstab_convdiff_matches_reference(ctx, golden_loader, case):
    """BiCGStab-DILU on the reference's convection-diffusion systems: with sequential sums the
    reference's solution, residual and iteration count bit for bit; with the default tree sums
    the iteration count within one at the reference's sor, and the reference's iterate within
    1e-9 relative FP64 residual at its iteration count."""
    g = golden_loader(case)
    csr = _csr_of(g)
    a, su = g.inp("a_convdiff"), g.inp("su_convdiff")
    sor, nsw = float(g.inp("sor")[0]), int(g.inp("nsw")[0])
    ref_iters = int(g.out("bicgstab", "iters")[0])
    ctx.set_reduction_order(fcap.REDUCE_SEQUENTIAL)
    try:
        rs = fcap.bicgstab(csr, a, su, g.inp("fi0"), sor=sor, nsw=nsw, ctx=ctx)
    finally:
        ctx.set_reduction_order(fcap.REDUCE_TREE)
    assert rs.info["iters"] == ref_iters
    np.testing.assert_array_equal(rs.fi, g.out("bicgstab", "fi"))
    np.testing.assert_array_equal(rs.res, g.out("bicgstab", "res"))
    r = fcap.bicgstab(csr, a, su, g.inp("fi0"), sor=sor, nsw=nsw, ctx=ctx)
    assert r.status == 0
    assert abs(r.info["iters"] - ref_iters) <= 1
    A = _dense(csr, a)
    bn = np.linalg.norm(su)
    r2 = fcap.bicgstab(csr, a, su, g.inp("fi0"), sor=1e-30, nsw=ref_iters, ctx=ctx)
    assert r2.status == fcap.FC_NOT_CONVERGED and r2.info["iters"] == ref_iters
    assert np.linalg.norm(A @ (r2.fi - g.out("bicgstab", "fi"))) / bn <= 1e-9


def test_solver_transcript_5x5(ctx):
    """tests/output.txt: iteration counts 6/5/5, res0 lines and the solutions (warm starts as in the reference)."""
    t = load_transcript()
    csr = fcap.CSR(np.array(t["ioffset"], np.int32), np.array(t["ja"], np.int32), np.array(t["diag"], np.int32),
                   np.zeros(0, np.int32), np.zeros(0, np.int32))
    r1 = fcap.bicgstab(csr, t["a1"], t["b1"], np.zeros(5), ctx=ctx, variant=fcap.VARIANT_TESTS)
    r2 = fcap.iccg(csr, t["a2"], t["b2"], r1.fi, ctx=ctx, variant=fcap.VARIANT_TESTS)
    r3 = fcap.dpcg(csr, t["a2"], t["b2"], r2.fi, ctx=ctx, variant=fcap.VARIANT_TESTS)
    assert (r1.info["iters"], r2.info["iters"], r3.info["iters"]) == (6, 5, 5)
    assert f"{r1.info['res0']:10.3E}" == " 2.903E+01"
    assert f"{r2.info['res0']:10.3E}" == " 3.725E+01"
    np.testing.assert_allclose(r1.fi, np.linalg.solve(np.array(t["a1"]).reshape(5, 5), t["b1"]), rtol=1e-12)
    np.testing.assert_allclose(r3.fi, np.linalg.solve(np.array(t["a2"]).reshape(5, 5), t["b2"]), rtol=1e-12)
    assert [f"{v:5.2f}" for v in r1.fi] == [f"{v:5.2f}" for v in t["xa1"]]


@pytest.mark.parametrize("solver", ["iccg", "dpcg", "bicgstab"])
def test_report_line_matches_reference(ctx, golden_loader, capfd, solver):
    """The one-line report (src/iccg.f90:174-175 and its dpcg/bicgstab twins): same text as the
    reference's line, character for character, up to the iteration count (+-1) and the last digit
    of the final residual."""
    import re

    g = golden_loader("hex8_perturbed")
    ref = str(g.out(solver, "report_line"))
    a, su = g.out(solver, "a"), g.out(solver, "su")
    ctx.set_report(True, "p")
    try:
        capfd.readouterr()
        getattr(fcap, solver)(_csr_of(g), a, su, g.inp("fi0"), sor=float(g.inp("sor")[0]),
                              nsw=int(g.inp("nsw")[0]), ctx=ctx)
        out = capfd.readouterr().out
    finally:
        ctx.set_report(False, "p")
    line = [ln for ln in out.splitlines() if "Solving for" in ln][-1]
    pat = r"^(.*Solving for p, Initial residual = )(.{10}), Final residual = (.{10}), No Iterations (\d+)$"
    mg, mr = re.match(pat, line), re.match(pat, ref)
    assert mg and mr, (line, ref)
    assert mg.group(1) == mr.group(1)                     # solver tag and spacing
    assert mg.group(2) == mr.group(2)                     # initial residual, %10.3E
    assert abs(int(mg.group(4)) - int(mr.group(4))) <= 1
    assert mg.group(3)[-4:] == mr.group(3)[-4:] or abs(float(mg.group(3)) / float(mr.group(3)) - 1) < 0.5


def test_early_exit_and_status_codes(ctx, golden_loader):
    g = golden_loader("hex4_uniform")
    csr = _csr_of(g)
    a = g.out(g.first, "a")
    x = np.random.default_rng(2).standard_normal(csr.diag.shape[0])
    su = O.spmv(O.CSR(csr.ioffset, csr.ja, csr.diag, csr.ij_slot, csr.ji_slot), a, x)
    r = fcap.iccg(csr, a, su, x, ctx=ctx)          # exact initial guess: res0 < 1e-13
    assert r.status == fcap.FC_EARLY_EXIT and r.info["iters"] == 0
    r = fcap.dpcg(csr, a, g.out(g.first, "su"), np.zeros_like(x), sor=1e-30, nsw=3, ctx=ctx)
    assert r.status == fcap.FC_NOT_CONVERGED and r.info["iters"] == 3
    bad = a.copy()
    bad[csr.diag[0] - 1] = np.nan
    with pytest.raises(fcap.FcError):
        fcap.iccg(csr, bad, g.out(g.first, "su"), np.zeros_like(x), ctx=ctx)


def test_structure_errors_are_reported(ctx):
    own1 = np.array([1, 1, 2], np.int32)
    nei1 = np.array([2, 2, 3], np.int32)            # duplicate pair (1,2)
    with pytest.raises(fcap.FcError) as e:
        fcap.create_csr_matrix_from_mesh_data(3, own1, nei1, ctx)
    assert e.value.status == -5
    with pytest.raises(fcap.FcError):
        fcap.create_csr_matrix_from_mesh_data(3, np.array([1], np.int32), np.array([7], np.int32), ctx)


# ------------------------------------------------------- pressure correction

@pytest.mark.parametrize("case", CALCP_CASES)
def test_calcp_bitwise_vs_reference(ctx, golden_loader, case):
    """fc_calcp_assemble against the reference's facefluxmass + calcp face loop."""
    g = golden_loader(case)
    geo = fcap.Geometry(*(g.out("calcp", k) for k in ("arx", "ary", "arz", "xf", "yf", "zf", "vol", "xc", "yc",
                                                      "zc", "facint")))
    csr = fcap.CSR(*(g.out("calcp", k) for k in ("ioffset", "ja", "diag", "ij_slot", "ji_slot")))
    out = fcap.calcp_assemble(g.mesh, geo, csr, {k: g.inp(k) for k in CALCP_FIELDS}, ctx=ctx)
    np.testing.assert_array_equal(out["flmass"], g.out("calcp", "flmass"))
    np.testing.assert_array_equal(out["a"], g.out("calcp", "a"))
    np.testing.assert_array_equal(out["su"], g.out("calcp", "su"))


def _mirror_cuts(m, og, seed):
    """O-C cuts on the boundary faces of the x = min plane, each joining the face's cell to the
    cell mirrored across the box (periodic-style pairs, S . d != 0)."""
    nif = m.n_inner
    nb = m.n_faces - nif
    xf = og.xf[nif:]
    faces = np.nonzero(np.abs(xf - xf.min()) < 1e-9)[0]
    # the cut faces must be consecutive face numbers: take the leading run
    run = faces[: np.argmax(np.diff(np.r_[faces, -10]) != 1) + 1]
    assert run.size >= 2 and nb > 0
    cells = m.owner[nif + run]
    xmax = og.xc.max() + og.xc.min()
    ctr = np.stack([og.xc, og.yc, og.zc], axis=1)
    tgt = np.stack([xmax - og.xc[cells], og.yc[cells], og.zc[cells]], axis=1)
    partner = np.array([int(np.argmin(((ctr - t) ** 2).sum(axis=1))) for t in tgt])
    rng = np.random.default_rng(seed)
    return {"ijl": cells, "ijr": partner, "foc": 0.3 + 0.4 * rng.random(run.size), "faces": nif + int(run[0])}


def test_calcp_oc_cuts_match_oracle(ctx):
    m = M.hex_box(5, perturb=0.2, seed=12)
    og = O.mesh_geometry(m)
    oc_csr = O.csr_build(m.n_cells, m.owner[:m.n_inner] + 1, m.neighbour + 1)
    rng = np.random.default_rng(4)
    n = m.n_cells
    f = {k: 0.5 + rng.random(n) for k in ("den", "apu", "apv", "apw")}
    f.update({k: rng.standard_normal(n) for k in ("u", "v", "w", "p")})
    f.update({k: rng.standard_normal((n, 3)) for k in ("dudx", "dvdx", "dwdx", "dpdx")})
    cuts = _mirror_cuts(m, og, 5)
    ref = O.calcp_assemble(m, og, oc_csr, f, oc=cuts)
    assert np.all(np.isfinite(ref["fmoc"])) and ref["fmoc"].size >= 2
    geo = fcap.Geometry(og.arx, og.ary, og.arz, og.xf, og.yf, og.zf, og.vol, og.xc, og.yc, og.zc, og.facint)
    csr = fcap.CSR(oc_csr.ioffset, oc_csr.ja, oc_csr.diag, oc_csr.ij_slot, oc_csr.ji_slot)
    out = fcap.calcp_assemble(m, geo, csr, f, oc=cuts, ctx=ctx)
    for k in ("a", "su", "flmass", "al", "ar", "fmoc"):
        np.testing.assert_array_equal(out[k], ref[k], err_msg=k)


def test_calcp_uniform_flow_closed_form(ctx):
    m, f, vel, grad = calcp_uniform_case()
    geo = fcap.mesh_geometry(m, ctx)
    csr = fcap.create_csr_matrix_from_mesh_data(m.n_cells, m.owner[:m.n_inner] + 1, m.neighbour + 1, ctx)
    n, nif = m.n_cells, m.n_inner
    for k, val in zip(("u", "v", "w"), vel):
        f[k] = np.full(n, val)
    for k in ("dudx", "dvdx", "dwdx"):
        f[k] = np.zeros((n, 3))
    f["p"] = grad[0] * geo.xc + grad[1] * geo.yc + grad[2] * geo.zc
    f["dpdx"] = np.tile(grad, (n, 1))
    out = fcap.calcp_assemble(m, geo, csr, f, ctx=ctx)
    S = np.stack([geo.arx[:nif], geo.ary[:nif], geo.arz[:nif]], axis=1)
    np.testing.assert_allclose(out["flmass"], f["den"][0] * S @ vel, rtol=0, atol=1e-12)
    assert abs(out["su"].sum()) < 1e-12


@pytest.mark.parametrize("case", CALCP_CASES)
def test_calcp_nonorth_bitwise_vs_reference(ctx, golden_loader, case):
    """fc_calcp_nonorth: fmcor against the reference's fluxmc, su against the oracle."""
    g = golden_loader(case)
    geo = fcap.Geometry(*(g.out("calcp", k) for k in ("arx", "ary", "arz", "xf", "yf", "zf", "vol", "xc", "yc",
                                                      "zc", "facint")))
    csr = fcap.CSR(*(g.out("calcp", k) for k in ("ioffset", "ja", "diag", "ij_slot", "ji_slot")))
    nif = g.mesh.n_inner
    su, fl, _ = fcap.calcp_nonorth(g.mesh, geo, csr, g.inp("den"), g.inp("apu"), g.inp("dpdx"), np.zeros(nif),
                                   ctx=ctx)
    np.testing.assert_array_equal(fl, g.out("calcp", "fmcor"))
    og = O.Geometry(*(g.out("calcp", k) for k in ("arx", "ary", "arz", "xf", "yf", "zf", "vol", "xc", "yc", "zc",
                                                  "facint")))
    fl0 = g.out("calcp", "flmass")
    osu, ofl, _, _ = O.calcp_nonorth(g.mesh, og, g.inp("den"), g.inp("apu"), g.inp("dpdx"), fl0)
    su2, fl2, _ = fcap.calcp_nonorth(g.mesh, geo, csr, g.inp("den"), g.inp("apu"), g.inp("dpdx"), fl0, ctx=ctx)
    np.testing.assert_array_equal(su, osu)
    np.testing.assert_array_equal(su2, osu)
    np.testing.assert_array_equal(fl2, ofl)


def test_calcp_nonorth_oc_cuts_match_oracle(ctx):
    m = M.hex_box(5, perturb=0.2, seed=12)
    og = O.mesh_geometry(m)
    oc_csr = O.csr_build(m.n_cells, m.owner[:m.n_inner] + 1, m.neighbour + 1)
    rng = np.random.default_rng(9)
    n, nif = m.n_cells, m.n_inner
    den, apu, gpp = 0.5 + rng.random(n), 0.5 + rng.random(n), rng.standard_normal((n, 3))
    fl0 = rng.standard_normal(nif)
    cuts = _mirror_cuts(m, og, 5)
    fm0 = rng.standard_normal(len(cuts["ijl"]))
    osu, ofl, ofm, _ = O.calcp_nonorth(m, og, den, apu, gpp, fl0, oc=cuts, fmoc=fm0)
    assert np.abs(ofm - fm0).max() > 1e-6
    geo = fcap.Geometry(og.arx, og.ary, og.arz, og.xf, og.yf, og.zf, og.vol, og.xc, og.yc, og.zc, og.facint)
    csr = fcap.CSR(oc_csr.ioffset, oc_csr.ja, oc_csr.diag, oc_csr.ij_slot, oc_csr.ji_slot)
    su, fl, fm = fcap.calcp_nonorth(m, geo, csr, den, apu, gpp, fl0, oc=cuts, fmoc=fm0, ctx=ctx)
    np.testing.assert_array_equal(su, osu)
    np.testing.assert_array_equal(fl, ofl)
    np.testing.assert_array_equal(fm, ofm)


@pytest.mark.parametrize("case", CALCP_CASES)
def test_calcp_correct_matches_oracle(ctx, golden_loader, case):
    """fc_calcp_correct with the reference's assembled matrix and random pp and gradient, plus
    O-C cuts on a perturbed box."""
    g = golden_loader(case)
    csr = fcap.CSR(*(g.out("calcp", k) for k in ("ioffset", "ja", "diag", "ij_slot", "ji_slot")))
    n = g.mesh.n_cells
    rng = np.random.default_rng(13)
    pp, gpp = rng.standard_normal(n), rng.standard_normal((n, 3))
    args = (g.out("calcp", "a"), pp, gpp, g.out("calcp", "vol"), g.inp("apu"), g.inp("apv"), g.inp("apw"), 0.2,
            n // 3, g.out("calcp", "flmass"), g.inp("u"), g.inp("v"), g.inp("w"), g.inp("p"))
    ref = O.calcp_correct(g.mesh, O.CSR(csr.ioffset, csr.ja, csr.diag, csr.ij_slot, csr.ji_slot), *args)
    out = fcap.calcp_correct(g.mesh, csr, *args, ctx=ctx)
    for k, (x, y) in enumerate(zip(out, ref)):
        np.testing.assert_array_equal(x, y, err_msg=str(k))


def test_calcp_correct_oc_cuts_and_errors(ctx):
    m = M.hex_box(5, perturb=0.2, seed=12)
    og = O.mesh_geometry(m)
    oc_csr = O.csr_build(m.n_cells, m.owner[:m.n_inner] + 1, m.neighbour + 1)
    csr = fcap.CSR(oc_csr.ioffset, oc_csr.ja, oc_csr.diag, oc_csr.ij_slot, oc_csr.ji_slot)
    rng = np.random.default_rng(14)
    n, nif = m.n_cells, m.n_inner
    cuts = _mirror_cuts(m, og, 5)
    noc = len(cuts["ijl"])
    a = rng.standard_normal(m.nnz)
    cell = [rng.standard_normal(n) for _ in range(4)]
    aps = [0.5 + rng.random(n) for _ in range(3)]
    args = (a, rng.standard_normal(n), rng.standard_normal((n, 3)), og.vol, *aps, 0.8, 0, rng.standard_normal(nif),
            *cell)
    kw = dict(oc=cuts, ar=rng.standard_normal(noc), fmoc=rng.standard_normal(noc))
    ref = O.calcp_correct(m, oc_csr, *args, **kw)
    out = fcap.calcp_correct(m, csr, *args, **kw, ctx=ctx)
    for k, (x, y) in enumerate(zip(out, ref)):
        np.testing.assert_array_equal(x, y, err_msg=str(k))
    bad = list(args)
    bad[8] = n                      # reference cell outside the mesh (0-based n)
    with pytest.raises(fcap.FcError):
        fcap.calcp_correct(m, csr, *bad, ctx=ctx)


def test_calcp_correct_consistent_with_velocity_correction(ctx):
    """On unit cubes with apu = apv = apw and pp linear: the flux correction a_ij (pp_N - pp_P) of
    the GPU-assembled matrix is rho times the interpolated velocity correction dotted with S."""
    m, f, _, grad = calcp_uniform_case()
    f["apv"] = f["apw"] = f["apu"]
    geo = fcap.mesh_geometry(m, ctx)
    csr = fcap.create_csr_matrix_from_mesh_data(m.n_cells, m.owner[:m.n_inner] + 1, m.neighbour + 1, ctx)
    n, nif = m.n_cells, m.n_inner
    rng = np.random.default_rng(6)
    f.update({k: rng.standard_normal(n) for k in ("u", "v", "w", "p")})
    f.update({k: np.zeros((n, 3)) for k in ("dudx", "dvdx", "dwdx", "dpdx")})
    a = fcap.calcp_assemble(m, geo, csr, f, ctx=ctx)["a"]
    pp = grad[0] * geo.xc + grad[1] * geo.yc + grad[2] * geo.zc
    fl0 = rng.standard_normal(nif)
    fl, _, u, v, w, p = fcap.calcp_correct(m, csr, a, pp, np.tile(grad, (n, 1)), geo.vol, f["apu"], f["apv"],
                                           f["apw"], 0.3, 5, fl0, f["u"], f["v"], f["w"], f["p"], ctx=ctx)
    o, q, lam = m.owner[:nif], m.neighbour, geo.facint
    du = np.stack([u - f["u"], v - f["v"], w - f["w"]], axis=1)
    duf = (1 - lam)[:, None] * du[o] + lam[:, None] * du[q]
    S = np.stack([geo.arx[:nif], geo.ary[:nif], geo.arz[:nif]], axis=1)
    np.testing.assert_allclose(fl - fl0, f["den"][0] * (duf * S).sum(axis=1), rtol=1e-12, atol=1e-14)
    assert p[5] == f["p"][5]


@pytest.mark.parametrize("case", ADJUST_CASES)
def test_adjust_mass_flow_bitwise_vs_reference(ctx, golden_loader, case):
    """fc_adjust_mass_flow against the reference's adjustMassFlow."""
    g = golden_loader(case)
    geo = fcap.Geometry(g.out("adjust", "arx"), g.out("adjust", "ary"), g.out("adjust", "arz"), *[None] * 8)
    args = (g.inp("flomas")[0], g.inp("den"), g.inp("u"), g.inp("v"), g.inp("w"), g.inp("su"), g.inp("fmi"))
    out = fcap.adjust_mass_flow(g.mesh, geo, *args, ctx=ctx)
    for k, x in zip(("su", "u", "v", "w", "fmo"), out):
        np.testing.assert_array_equal(x, g.out("adjust", k), err_msg=k)


def test_adjust_mass_flow_long_outlet_matches_oracle(ctx):
    """An outlet of 900 faces (the ordered sum runs over 15 loads of 64) and cells owning an
    inlet and an outlet face at once (a box one cell long in x)."""
    m = M.hex_box(1, 30, 30, perturb=0.1, seed=3)
    m.patches = [(t, nf, st) for t, (_, nf, st) in zip(["inlet", "outlet", "wall", "wall", "wall", "wall"],
                                                       m.patches)]
    og = O.mesh_geometry(m)
    n, ntot = m.n_cells, m.n_cells + m.n_boundary
    ninl = int(O.boundary_groups(m)[0])
    rng = np.random.default_rng(21)
    args = (1.7, 1 + 0.1 * rng.random(ntot), 1 + 0.2 * rng.standard_normal(ntot), rng.standard_normal(ntot),
            rng.standard_normal(ntot), rng.standard_normal(n), rng.random(ninl))
    ref = O.adjust_mass_flow(m, og, *args)
    assert ref[4].size == 900
    geo = fcap.Geometry(og.arx, og.ary, og.arz, og.xf, og.yf, og.zf, og.vol, og.xc, og.yc, og.zc, og.facint)
    out = fcap.adjust_mass_flow(m, geo, *args, ctx=ctx)
    for k, (x, y) in enumerate(zip(out, ref)):
        np.testing.assert_array_equal(x, y, err_msg=str(k))


def test_adjust_mass_flow_with_device_resident_fields(ctx, golden_loader):
    """Floating-point arrays may be device memory: the library copies them on the device.  The
    fields of fc_adjust_mass_flow in hipMalloc'd buffers give the reference's bits as well."""
    import ctypes as C
    hip = C.CDLL("libamdhip64.so")
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    hip.hipFree.argtypes = [C.c_void_p]
    g = golden_loader("hex5_adjust")
    m = g.mesh
    n, ntot = m.n_cells, m.n_cells + m.n_boundary
    bnd = fcap.boundary_groups(m)
    host = {k: np.ascontiguousarray(g.inp(k), np.float64) for k in ("den", "u", "v", "w", "su", "fmi")}
    for k in ("arx", "ary", "arz"):
        host[k] = np.ascontiguousarray(g.out("adjust", k), np.float64)
    host["fmo"] = np.zeros(int(bnd[2]))
    dev = {}
    try:
        for k, a in host.items():
            p = C.c_void_p()
            assert hip.hipMalloc(C.byref(p), max(a.nbytes, 8)) == 0
            dev[k] = p
            assert hip.hipMemcpy(p, a.ctypes.data, a.nbytes, 1) == 0        # host to device
        dp = lambda k: C.cast(dev[k], C.POINTER(C.c_double))  # noqa: E731
        own1 = (m.owner.astype(np.int64) + 1).astype(np.int32)
        rc = ctx.L.fc_adjust_mass_flow(ctx.h, n, ntot, m.n_faces, own1.ctypes.data_as(C.POINTER(C.c_int)),
                                       dp("arx"), dp("ary"), dp("arz"), int(bnd[0]), int(bnd[1]), dp("fmi"),
                                       int(bnd[2]), int(bnd[3]), n + int(bnd[0]), float(g.inp("flomas")[0]),
                                       dp("den"), dp("u"), dp("v"), dp("w"), dp("su"), dp("fmo"))
        assert rc == fcap.FC_OK, ctx.L.fc_last_error(ctx.h)
        for k in ("su", "u", "v", "w", "fmo"):
            out = np.zeros_like(host[k])
            assert hip.hipMemcpy(out.ctypes.data, dev[k], out.nbytes, 2) == 0   # device to host
            np.testing.assert_array_equal(out, g.out("adjust", k), err_msg=k)
    finally:
        for p in dev.values():
            hip.hipFree(p)


def test_step_entry_points_reject_bad_arguments(ctx, golden_loader):
    """The pressure-correction step's entry points check their sizes and ranges before any kernel
    runs, and the tuning setters their values."""
    import ctypes as C
    g = golden_loader("hex5_adjust")
    m = g.mesh
    geo = fcap.Geometry(g.out("adjust", "arx"), g.out("adjust", "ary"), g.out("adjust", "arz"), *[None] * 8)
    args = (g.inp("flomas")[0], g.inp("den"), g.inp("u"), g.inp("v"), g.inp("w"), g.inp("su"), g.inp("fmi"))
    n, ntot = m.n_cells, m.n_cells + m.n_boundary
    own1 = (m.owner.astype(np.int64) + 1).astype(np.int32)
    dp = lambda x: np.ascontiguousarray(x, np.float64).ctypes.data_as(C.POINTER(C.c_double))  # noqa: E731
    ip = lambda x: np.ascontiguousarray(x, np.int32).ctypes.data_as(C.POINTER(C.c_int))  # noqa: E731
    u, v, w, su, fmo = (np.array(x, np.float64) for x in (g.inp("u"), g.inp("v"), g.inp("w"), g.inp("su"),
                                                           np.zeros(64)))
    bnd = fcap.boundary_groups(m)
    # outlet values past numTotal
    rc = ctx.L.fc_adjust_mass_flow(ctx.h, n, ntot, m.n_faces, ip(own1), dp(geo.arx), dp(geo.ary), dp(geo.arz),
                                   int(bnd[0]), int(bnd[1]), dp(g.inp("fmi")), int(bnd[2]), int(bnd[3]), ntot - 1,
                                   1.0, dp(g.inp("den")), dp(u), dp(v), dp(w), dp(su), dp(fmo))
    assert rc == fcap.FC_ERR_ARGUMENT
    # inlet faces past the faces
    rc = ctx.L.fc_adjust_mass_flow(ctx.h, n, ntot, m.n_faces, ip(own1), dp(geo.arx), dp(geo.ary), dp(geo.arz),
                                   int(bnd[0]), m.n_faces, dp(g.inp("fmi")), int(bnd[2]), int(bnd[3]), n,
                                   1.0, dp(g.inp("den")), dp(u), dp(v), dp(w), dp(su), dp(fmo))
    assert rc == fcap.FC_ERR_ARGUMENT
    # the valid call still works afterwards
    out = fcap.adjust_mass_flow(m, geo, *args, ctx=ctx)
    np.testing.assert_array_equal(out[0], g.out("adjust", "su"))
    # corrector source with a structure that does not match numInnerFaces
    c = O.csr_build(m.n_cells, m.owner[:m.n_inner] + 1, m.neighbour + 1)
    rc = ctx.L.fc_calcp_nonorth(ctx.h, n, m.n_inner - 1, ip(own1), ip(m.neighbour + 1), *[dp(np.zeros(m.n_faces))] * 11,
                                dp(np.ones(n)), dp(np.ones(n)), dp(np.zeros(3 * n)), 0, 0, ip([0]), ip([0]),
                                dp([0.0]), ip(c.ioffset), ip(c.ja), ip(c.diag), ip(c.ij_slot), ip(c.ji_slot),
                                m.nnz, dp(np.zeros(n)), dp(np.zeros(m.n_inner)), dp([0.0]))
    assert rc == fcap.FC_ERR_ARGUMENT
    # reference cell outside the mesh is covered by test_calcp_correct_oc_cuts_and_errors; setters
    for bad in ((-1, 0.8), (9, 0.8), (3, 0.0), (3, 2.0)):
        with pytest.raises(fcap.FcError):
            ctx.set_fcg_smoothing(*bad)
    for bad_mode in (1, 4, -1):   # 1 was a schedule this library no longer has
        with pytest.raises(fcap.FcError):
            ctx.set_sweep_mode(bad_mode)
    for bad_waves in (-1, 1 << 20):
        with pytest.raises(fcap.FcError):
            ctx.set_sweep_waves(bad_waves)
    ctx.set_fcg_smoothing()
    ctx.set_sweep_waves(0)
    ctx.set_sweep_mode(fcap.SWEEP_DEFAULT)


# ---------------------------------------------------------------- Gauss gradient

@pytest.mark.parametrize("case", GRAD_CASES)
@pytest.mark.parametrize("nigrad", [1, 2])
def test_grad_gauss_bitwise_vs_reference(ctx, golden_loader, case, nigrad):
    g = golden_loader(case)
    s = f"grad{nigrad}"
    geo = fcap.Geometry(*(g.out(s, k) for k in ("arx", "ary", "arz", "xf", "yf", "zf", "vol", "xc", "yc", "zc",
                                                "facint")))
    out = fcap.grad_gauss(g.mesh, geo, g.inp("u"), nigrad, ctx=ctx)
    for a, k in zip(out, ("dudx", "dudy", "dudz")):
        np.testing.assert_array_equal(a, g.out(s, k), err_msg=k)


@pytest.mark.parametrize("legs", [1, 7, 8, 9, 16, 41])
@pytest.mark.parametrize("shuffled", [False, True])
def test_grad_gauss_rows_of_any_length(ctx, legs, shuffled):
    """Rows of up to 41 faces (the row kernel takes eight a turn), faces in canonical order and
    shuffled, one to three passes: the oracle's bits.  The geometry is arbitrary numbers."""
    rng = np.random.default_rng(legs)
    n = legs + 1
    pairs = [(0, i) for i in range(1, n)] + [(i, i + 1) for i in range(1, n - 1)]
    order = rng.permutation(len(pairs)) if shuffled else np.arange(len(pairs))
    own, nei = np.array(pairs, np.int32)[order].T
    nif, nb = len(pairs), 3
    owner = np.concatenate([own, [0, 0, n - 1]]).astype(np.int32)
    m = M.PolyMesh(np.zeros((3, 3)), np.arange(0, 3 * (nif + nb) + 1, 3, dtype=np.int32),
                   np.zeros(3 * (nif + nb), np.int32), owner, np.ascontiguousarray(nei), n,
                   [("inlet", 1, nif), ("wall", 2, nif + 1)])
    face = lambda: rng.standard_normal(nif + nb)  # noqa: E731
    cell = lambda: rng.standard_normal(n)  # noqa: E731
    geo = fcap.Geometry(face(), face(), face(), face(), face(), face(), 0.5 + rng.random(n), cell(), cell(), cell(),
                        rng.random(nif))
    u = rng.standard_normal(n + nb)
    for nigrad in (1, 2, 3):
        out = fcap.grad_gauss(m, geo, u, nigrad, ctx=ctx)
        ref = O.grad_gauss(m, geo, u, nigrad)
        for a, b, k in zip(out, ref, ("dudx", "dudy", "dudz")):
            np.testing.assert_array_equal(a, b, err_msg=f"{k} nigrad={nigrad}")


def test_grad_gauss_oc_cuts_match_oracle(ctx):
    m = M.hex_box(5, perturb=0.2, seed=12)
    og = O.mesh_geometry(m)
    cuts = _mirror_cuts(m, og, 7)
    rng = np.random.default_rng(8)
    u = rng.standard_normal(m.n_cells + m.n_boundary)
    geo = fcap.Geometry(og.arx, og.ary, og.arz, og.xf, og.yf, og.zf, og.vol, og.xc, og.yc, og.zc, og.facint)
    for nig in (1, 3):
        ref = O.grad_gauss(m, og, u, nig, oc=cuts)
        out = fcap.grad_gauss(m, geo, u, nig, oc=cuts, ctx=ctx)
        for a, b, k in zip(out, ref, ("dudx", "dudy", "dudz")):
            np.testing.assert_array_equal(a, b, err_msg=f"{k} nigrad={nig}")


# ------------------------------------------------------- PISO assembly, bpres, velocity BCs

def _calcp_geo_csr(g):
    geo = fcap.Geometry(*(g.out("calcp", k) for k in ("arx", "ary", "arz", "xf", "yf", "zf", "vol", "xc", "yc", "zc",
                                                      "facint")))
    csr = fcap.CSR(*(g.out("calcp", k) for k in ("ioffset", "ja", "diag", "ij_slot", "ji_slot")))
    return geo, csr


@pytest.mark.parametrize("case", CALCP_CASES)
def test_piso_assemble_bitwise_vs_reference(ctx, golden_loader, case):
    """PISO's face loop around facefluxmass_piso on the GPU: flmass, a and su are the reference's
    bits (golden vectors of ref_flux_driver; the reference-pressure pin, which the host entry
    point leaves to the caller, applied to the GPU result on the host first)."""
    g = golden_loader(case)
    geo, csr = _calcp_geo_csr(g)
    out = fcap.piso_assemble(g.mesh, geo, csr, {k: g.inp(k) for k in PISO_FIELDS}, ctx=ctx)
    np.testing.assert_array_equal(out["flmass"], g.out("piso", "flmass"))
    a, su = out["a"].copy(), out["su"].copy()
    r = int(g.out("piso", "pref_cell")[0]) - 1
    a[csr.ioffset[r] - 1:csr.ioffset[r + 1] - 1] = 0.0
    a[csr.diag[r] - 1] = 1.0
    su[r] = g.inp("p")[r]
    np.testing.assert_array_equal(a, g.out("piso", "a"))
    np.testing.assert_array_equal(su, g.out("piso", "su"))


@pytest.mark.parametrize("case", BC_CASES)
def test_bpres_and_velocity_bc_bitwise_vs_reference(ctx, golden_loader, case):
    """bpres (stage 1 copies owner values, stage 2 extrapolates wall and pressure-outlet values)
    and correctBoundaryConditionsVelocity (outlet scaled to flomas in outlet order, symmetry
    projected) on the GPU: the reference's bits on meshes with every boundary group."""
    g = golden_loader(case)
    m = g.mesh
    geo = fcap.mesh_geometry(m, ctx)
    p1 = fcap.bpres(m, geo, g.inp("p"), None, 1, ctx=ctx)
    np.testing.assert_array_equal(p1, g.out("bc", "p1"))
    p2 = fcap.bpres(m, geo, p1, g.inp("dpdx"), 2, ctx=ctx)
    np.testing.assert_array_equal(p2, g.out("bc", "p2"))
    u, v, w, fmo = fcap.correct_velocity_bc(m, geo, g.inp("flomas")[0], g.inp("den"), g.inp("u"), g.inp("v"),
                                            g.inp("w"), ctx=ctx)
    for k, x in (("u", u), ("v", v), ("w", w), ("fmo", fmo)):
        np.testing.assert_array_equal(x, g.out("bc", k), err_msg=k)


def test_bpres_oc_cuts_match_oracle(ctx, golden_loader):
    """bpres with O-C cuts after the pressure-outlet values: stage 1 copies the owners' values,
    stage 2 extrapolates with the face centre the reference indexes by the cut number
    (bpres.f90:140-142); bitwise the oracle."""
    g = golden_loader("hex5_bc")
    m = g.mesh
    geo = fcap.mesh_geometry(m, ctx)
    noc, oc0 = 5, m.n_inner + 3          # five boundary faces treated as cuts
    rng = np.random.default_rng(4)
    p = rng.standard_normal(m.n_cells + m.n_boundary + noc)
    dpdx = rng.standard_normal((m.n_cells, 3))
    og = O.Geometry(*(getattr(geo, k) for k in ("arx", "ary", "arz", "xf", "yf", "zf", "vol", "xc", "yc", "zc",
                                                "facint")))
    for stage, dg in ((1, None), (2, dpdx)):
        got = fcap.bpres(m, geo, p, dg, stage, noc=noc, oc_faces_start=oc0, ctx=ctx)
        want = O.bpres(m, og, p, dg, stage, noc=noc, oc_faces_start=oc0)
        np.testing.assert_array_equal(got, want, err_msg=f"stage {stage}")
        assert not np.array_equal(got, p)
        p = got


@pytest.mark.parametrize("mesh", ["hex32", "hex24_graded", "tet12"])
def test_part_sweeps_bitwise_on_multi_part_meshes(ctx, mesh):
    """Meshes of several parts (hex 32^3: 16 pencils; graded 24^3: 9; Kuhn tets 12^3: 3 runs of
    4,096 rows): the part-wise sweeps (inputs inside a part through LDS, across parts through
    global memory) give the DIC and DILU sweeps of the oracle bit for bit, as the other schedules
    do."""
    m = {"hex32": lambda: M.hex_box(32, perturb=0.2, seed=3),
         "hex24_graded": lambda: M.hex_box(24, perturb=0.2, seed=4, grade_axis=0, grade_ratio=1.2,
                                           grade_max_aspect=50.0),
         "tet12": lambda: M.tet_box(12, grade_axis=1, grade_ratio=1.1)}[mesh]()
    geo = O.mesh_geometry(m)
    oc = O.csr_build(m.n_cells, m.owner[:m.n_inner] + 1, m.neighbour + 1)
    csr = fcap.CSR(oc.ioffset, oc.ja, oc.diag, oc.ij_slot, oc.ji_slot)
    a, _ = O.laplacian(m, geo, oc, np.full(m.n_cells, -1.0), np.zeros(m.n_cells + m.n_boundary),
                       np.zeros(m.n_cells))
    u, v, w = W.taylor_green(geo.xc, geo.yc, geo.zc)
    ac = O.convdiff(m, geo, oc, np.full(m.n_cells, 1e-3), O.face_flux_central(m, geo, u, v, w), 0.7)
    r = np.random.default_rng(5).standard_normal(m.n_cells)
    try:
        for mat, dilu in ((a, False), (ac, True)):
            d_ref = O.dilu_pivots(oc, mat) if dilu else O.dic_pivots(oc, mat)
            ref = O.lu_apply(oc, mat, d_ref, r)
            for mode in (fcap.SWEEP_PARTS, fcap.SWEEP_DEPENDENT):
                ctx.set_sweep_mode(mode)
                d = fcap.dilu_pivots(csr, mat, ctx) if dilu else fcap.dic_pivots(csr, mat, ctx)
                np.testing.assert_array_equal(d, d_ref, err_msg=f"pivots, mode {mode}")
                np.testing.assert_array_equal(fcap.lu_apply(csr, mat, d, r, ctx), ref, err_msg=f"mode {mode}")
    finally:
        ctx.set_sweep_mode(fcap.SWEEP_DEFAULT)


def _renumbered(m, order):
    """The mesh with cell `order[k]` numbered k (faces put back into upper-triangular order)."""
    new = np.empty(m.n_cells, np.int64)
    new[order] = np.arange(m.n_cells)
    nif = m.n_inner
    nodes = m.face_nodes.reshape(m.n_faces, -1)
    return M._canonical_polymesh(m.points, m.n_cells, new[m.owner[:nif]], new[m.neighbour], nodes[:nif],
                                 new[m.owner[nif:]], nodes[nif:],
                                 np.repeat(np.arange(len(m.patches)), [p[1] for p in m.patches]),
                                 [p[0] for p in m.patches])


def _part_meshes():
    # pencils: full and ragged line and sheet blocks, one sheet, one line, one cell, thin sheets
    for dims in ((9, 7, 5), (16, 16, 16), (17, 65, 1), (300, 1, 1), (5, 130, 1), (3, 2, 70), (70, 9, 17), (1, 1, 1),
                 (33, 64, 2), (12, 1, 40)):
        yield "box_%dx%dx%d" % dims, M.hex_box(*dims)
    # two blocks numbered one after the other, a sheet of each size: two stacks
    m = M.hex_box(24, 20, 12)
    c = np.arange(m.n_cells)
    i = c % 24
    yield "two_blocks", _renumbered(m, np.concatenate([c[i < 9], c[i >= 9]]))
    # numberings without such runs: consecutive parts (z fastest in tiles); scattered rows, which
    # read too little of their own part and take the row-wise sweeps
    x, y, z = i, (c // 24) % 20, c // 480
    yield "tiles", _renumbered(m, np.lexsort((x % 4, z % 4, y % 4, x // 4, y // 4, z // 4)))
    yield "scattered", _renumbered(m, np.random.default_rng(4).permutation(m.n_cells))


@pytest.mark.gpu
@pytest.mark.parametrize("name,m", list(_part_meshes()), ids=lambda v: v if isinstance(v, str) else "")
def test_part_sweeps_bitwise_over_numberings(ctx, name, m):
    """The sweeps the default chooses over every form of parts -- pencils with ragged line and sheet
    blocks, several stacks, consecutive runs -- and over scattered rows give the oracle's DIC and DILU sweeps bit for bit, and the
    FP32 sweeps inside the mixed solver the same iterates as one launch per level."""
    geo = O.mesh_geometry(m)
    csr = O.csr_build(m.n_cells, m.owner[:m.n_inner] + 1, m.neighbour + 1)
    rng = np.random.default_rng(11)
    su = rng.uniform(-1, 1, m.n_cells)
    a, _ = O.laplacian(m, geo, csr, np.full(m.n_cells, -1.0), np.zeros(m.n_cells + m.n_boundary), su)
    r = rng.uniform(-1, 1, m.n_cells)
    d = O.dic_pivots(csr, a)
    np.testing.assert_array_equal(fcap.lu_apply(csr, a, d, r, ctx), O.lu_apply(csr, a, d, r), err_msg=name)
    skew = a * rng.uniform(0.8, 1.2, a.shape[0])
    dl = O.dilu_pivots(csr, skew)
    np.testing.assert_array_equal(fcap.lu_apply(csr, skew, dl, r, ctx), O.lu_apply(csr, skew, dl, r), err_msg=name)
    s = fcap.System(m, ctx)
    out = []
    try:
        for mode in (fcap.SWEEP_PARTS, fcap.SWEEP_LEVELS):
            ctx.set_sweep_mode(mode)
            s.assemble_laplacian(np.full(m.n_cells, -1.0), None, su)
            s.set_solution(np.zeros(m.n_cells))
            s.solve(fcap.METHOD_ICCG_MIXED, fcap.STOP_L2, 1e-8, 500)
            out.append(s.solution())
    finally:
        ctx.set_sweep_mode(fcap.SWEEP_DEFAULT)
        s.close()
    np.testing.assert_array_equal(out[0], out[1], err_msg=name)


@pytest.mark.gpu
@pytest.mark.parametrize("waves", [0, 1, 2, 7, 8, 9, 300])
@pytest.mark.parametrize("mesh", ["tets", "box", "row"])
def test_row_sweeps_bitwise_over_wave_counts(ctx, mesh, waves):
    """The row-wise dependency-driven sweeps with fewer, as many and more waves than block
    counters, and more than blocks: pairs of sweeps one after the other inside DIC-PCG, BiCGStab
    and the mixed solver give the iterates of one launch per level bit for bit."""
    m = {"tets": lambda: M.tet_box(6, permute_seed=3), "box": lambda: M.hex_box(13, 11, 7, perturb=0.1, seed=1),
         "row": lambda: M.hex_box(70, 1, 1)}[mesh]()
    su = np.random.default_rng(5).uniform(-1, 1, m.n_cells)
    s = fcap.System(m, ctx)
    out = {}
    try:
        ctx.set_sweep_waves(waves)
        for mode in (fcap.SWEEP_DEPENDENT, fcap.SWEEP_LEVELS):
            ctx.set_sweep_mode(mode)
            for method in (fcap.METHOD_ICCG, fcap.METHOD_BICGSTAB, fcap.METHOD_ICCG_MIXED):
                s.assemble_laplacian(np.full(m.n_cells, -1.0), None, su)
                s.set_solution(np.zeros(m.n_cells))
                s.solve(method, fcap.STOP_L2, 1e-8, 500)
                out.setdefault(method, []).append(s.solution())
    finally:
        ctx.set_sweep_waves(0)
        ctx.set_sweep_mode(fcap.SWEEP_DEFAULT)
        s.close()
    for method, (a, b) in out.items():
        np.testing.assert_array_equal(a, b, err_msg=str(method))


@pytest.mark.gpu
@pytest.mark.parametrize("method", ["ICCG", "DPCG", "BICGSTAB", "ICCG_MIXED", "BICGSTAB_MIXED", "FCG_JACOBI"])
def test_solves_that_end_before_and_after_the_graph(ctx, method):
    """Solves of 1 to 12 iterations -- launched one by one, ending as the graph of iterations is set
    up, and replayed from it -- stop at their limit and give the iterates of launches alone."""
    m = M.hex_box(13, 11, 9, perturb=0.1, seed=2)
    su = np.random.default_rng(6).uniform(-1, 1, m.n_cells)
    s = fcap.System(m, ctx)
    try:
        for mode in (fcap.SWEEP_PARTS, fcap.SWEEP_DEPENDENT, fcap.SWEEP_LEVELS):
            ctx.set_sweep_mode(mode)
            for nsw in range(1, 13):
                out = []
                for graphs in (True, False):
                    ctx.set_graphs(graphs)
                    s.assemble_laplacian(np.full(m.n_cells, -1.0), None, su)
                    s.set_solution(np.zeros(m.n_cells))
                    _, info = s.solve(getattr(fcap, "METHOD_" + method), fcap.STOP_L2, 1e-15, nsw)
                    assert info["iters"] == nsw
                    out.append(s.solution())
                np.testing.assert_array_equal(out[0], out[1], err_msg=f"mode {mode}, nsw {nsw}")
    finally:
        ctx.set_graphs(True)
        ctx.set_sweep_mode(fcap.SWEEP_DEFAULT)
        s.close()


def _structure(n, lo, hi):
    """(ioffset, ja, diag), 1-based, of n rows coupled in the pairs (lo, hi)."""
    i = np.arange(n)
    key = np.unique(np.concatenate([lo, hi, i]) * n + np.concatenate([hi, lo, i]))
    row, col = key // n, key % n
    one = lambda x: np.ascontiguousarray(x + 1, np.int32)  # noqa: E731
    return one(np.concatenate([[0], np.cumsum(np.bincount(row))])), one(col), one(np.flatnonzero(row == col))


def _hubs(groups, mirrored):
    """Rows in groups of seven, the last of a group coupled to the six before it, and every row to the
    one 200 on: seven entries in a strict lower triangle's widest row and two in the upper's, or
    mirrored the other way round."""
    n = 7 * groups
    i = np.arange(n)
    lo, hi = np.concatenate([np.stack([i[:-200], i[200:]])] + [np.stack([i[k::7], i[6::7]]) for k in range(6)], axis=1)
    return _structure(n, n - 1 - lo, n - 1 - hi) if mirrored else _structure(n, lo, hi)


def _shuffled(structure, run):
    """The structure with its rows in random order within runs of consecutive ones."""
    ioffset, ja, diag = structure
    n = len(diag)
    new = np.empty(n, np.int64)
    new[np.lexsort((np.random.default_rng(n).random(n), np.arange(n) // run))] = np.arange(n)
    return _structure(n, new[np.repeat(np.arange(n), np.diff(ioffset))], new[ja - 1])


def _wide_structures():
    import part_model as P
    yield "four", P.stencil((24, 20, 40), P.STEPS6[:4]), 4, 4
    yield "six", P.stencil((24, 20, 40), P.STEPS6), 8, 8
    yield "eight", P.stencil((20, 17, 41), P.STEPS8), 8, 8
    yield "four_runs", _shuffled(P.stencil((90, 150, 1), P.STEPS6[:2]), 200), 4, 4
    yield "eight_runs", _shuffled(P.stencil((20, 18, 40), P.STEPS6[:4]), 150), 8, 8
    yield "hubs", _hubs(2000, False), 8, 3
    yield "mirrored_hubs", _hubs(2000, True), 3, 8


@pytest.mark.gpu
@pytest.mark.parametrize("name,structure,wf,wb", list(_wide_structures()), ids=lambda v: v if isinstance(v, str) else "")
def test_part_sweeps_bitwise_over_row_widths(ctx, name, structure, wf, wb):
    """Part-wise sweeps whose rows have four to eight entries in a triangle, the same width in both or
    not, pencils and runs, in several parts each longer than the ring in LDS: the oracle's DIC and DILU sweeps bit
    for bit.  The schedule chosen is the part-wise one by the rule restated here."""
    import part_model as P
    ioffset, ja, diag = structure
    oc = O.CSR(ioffset, ja, diag, np.zeros(0, np.int32), np.zeros(0, np.int32))
    zero = ioffset - 1, ja - 1, diag - 1
    low, up = (zero[2] - zero[0][:-1]).max(), (zero[0][1:] - 1 - zero[2]).max()
    assert [3 if w <= 3 else 4 if w <= 4 else 8 for w in (low, up)] == [wf, wb] and max(low, up) <= 8
    s = P.Schedule(*zero, *(P.pencil_parts(*zero) or P.run_parts(*zero)))
    for upper, width in ((False, wf), (True, wb)):
        s.codes(upper, width, 1024)
        assert s.inside >= 0.5, (name, s.inside)
    assert s.nparts >= 3 and np.diff(s.win).max() > 16
    n = len(diag)
    rng = np.random.default_rng(7)
    row = np.repeat(np.arange(n), np.diff(ioffset))
    key = np.minimum(row, ja - 1) * n + np.maximum(row, ja - 1)
    a = -rng.uniform(0.5, 1.0, ja.size)[np.unique(key, return_inverse=True)[1]]
    a[zero[2]] = 20.0
    r = rng.standard_normal(n)
    csr = fcap.CSR(ioffset, ja, diag, oc.ij_slot, oc.ji_slot)
    for mat, pivots in ((a, O.dic_pivots), (a * rng.uniform(0.8, 1.2, a.size), O.dilu_pivots)):
        d = pivots(oc, mat)
        np.testing.assert_array_equal(fcap.lu_apply(csr, mat, d, r, ctx), O.lu_apply(oc, mat, d, r), err_msg=name)


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["box", "tets"])
def test_part_sweeps_of_wide_rows_in_the_solvers(ctx, name):
    """Meshes shuffled within runs of 300 cells (up to six neighbours before a cell; up to four in
    the tets): the solvers' FP64 and FP32 part-wise sweeps give the iterates of one launch per level."""
    m = M.hex_box(24, 20, 40) if name == "box" else M.tet_box(14)
    c = np.arange(m.n_cells)
    m = _renumbered(m, np.lexsort((np.random.default_rng(3).random(m.n_cells), c // 300)))
    su = np.random.default_rng(8).uniform(-1, 1, m.n_cells)
    s = fcap.System(m, ctx)
    out = {}
    try:
        for mode in (fcap.SWEEP_PARTS, fcap.SWEEP_LEVELS):
            ctx.set_sweep_mode(mode)
            for method in (fcap.METHOD_ICCG, fcap.METHOD_ICCG_MIXED, fcap.METHOD_BICGSTAB_MIXED):
                s.assemble_laplacian(np.full(m.n_cells, -1.0), None, su)
                s.set_solution(np.zeros(m.n_cells))
                s.solve(method, fcap.STOP_L2, 1e-8, 500)
                out.setdefault(method, []).append(s.solution())
    finally:
        ctx.set_sweep_mode(fcap.SWEEP_DEFAULT)
        s.close()
    for method, (x, y) in out.items():
        np.testing.assert_array_equal(x, y, err_msg=str(method))


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [(128, 64, 64), (129, 64, 64)])
@pytest.mark.parametrize("method", ["BICGSTAB", "BICGSTAB_MIXED", "ICCG_MIXED"])
def test_solves_around_the_limit_of_direct_sums(ctx, dims, method):
    """524,288 and 528,384 rows: up to the first the vector kernels add the product's partials (one or
    two sums) themselves, beyond it a launch of its own does; the residual reached is the one asked for."""
    import scipy.sparse as sp
    m = M.hex_box(*dims)
    n = m.n_cells
    su = np.random.default_rng(9).uniform(-1, 1, n)
    su -= su.mean()
    s = fcap.System(m, ctx)
    try:
        s.assemble_laplacian(np.full(n, -1.0), None, su)
        rc, info = s.solve(getattr(fcap, "METHOD_" + method), fcap.STOP_L2, 1e-6, 2000)
        assert rc == fcap.FC_OK, (rc, info)
        A = sp.csr_matrix((s.get("a"), s.get("ja") - 1, s.get("ioffset") - 1), shape=(n, n))
        b = s.get("su")
        # the recurrence's residual and the true one part by rounding: at most iterations x eps x |A||x|
        rel = np.linalg.norm(b - A @ s.solution()) / np.linalg.norm(b)
        assert rel < 1e-6 * 1.01, (rel, info)
    finally:
        s.close()


@pytest.mark.gpu
def test_row_sweeps_of_several_contexts_at_once():
    """Three contexts in threads of their own, each with a wave for every 64 rows of its row-wise
    sweeps -- together more than the GPU holds, so none has all of its workgroups running: the
    iterates of a solve alone."""
    import threading
    m = M.tet_box(40, permute_seed=3)
    su = np.random.default_rng(4).uniform(-1, 1, m.n_cells)
    contexts = [fcap.Context(0) for _ in range(3)]
    systems, out, errors = [], [None] * 3, []
    try:
        for c in contexts:
            c.set_sweep_mode(fcap.SWEEP_DEPENDENT)
            c.set_sweep_waves(65536)
            s = fcap.System(m, c)
            s.assemble_laplacian(np.full(m.n_cells, -1.0), None, su)
            systems.append(s)

        def solve(k):
            try:
                systems[k].set_solution(np.zeros(m.n_cells))
                systems[k].solve(fcap.METHOD_ICCG, fcap.STOP_L2, 1e-15, 40)
                out[k] = systems[k].solution()
            except Exception as e:   # noqa: BLE001
                errors.append(repr(e))

        solve(0)
        alone = out[0]
        threads = [threading.Thread(target=solve, args=(k,)) for k in range(3)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors
        for x in out:
            np.testing.assert_array_equal(x, alone)
    finally:
        for s in systems:
            s.close()
        for c in contexts:
            c.close()
