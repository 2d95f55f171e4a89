"""Parity of the HIP engine (through the C ABI) with the CPU oracle.

Bars: stencil coefficients, branch codes, IB classification and the reference
multigrid primitives bit-exact; operator applications to rounding; pressure
increment phi within relative L2 1e-8 of the oracle's FP64 GMRES solution after
null-space removal, max|div u| <= 1e-8, and the projected fields consistent with
the oracle's projection of the engine's own phi to rounding.
"""
import numpy as np
import pytest

from oracle import oracle as O
from vfs_v3p2_amd import cases

pytestmark = pytest.mark.gpu

PHI_TOL = 1e-8
DIV_TOL = 1e-8


def affine_case(nx=10, ny=9, nz=8, seed=0):
    """Non-periodic grid under a full (sheared) affine map with a random flux field
    whose boundary faces carry no flux (a consistent Neumann problem)."""
    M = np.array([[1.0, 0.35, -0.2], [0.15, 0.8, 0.1], [-0.25, 0.3, 1.2]])
    ii, jj, kk = np.meshgrid(np.arange(nx + 1) / nx, np.arange(ny + 1) / ny, np.arange(nz + 1) / nz, indexing="xy")
    N = np.stack([ii, jj, kk], -1).transpose(2, 0, 1, 3) @ M.T
    co = cases.dmda_coords(N)
    f = cases.form_metrics(co, (0, 0, 0))
    f["nvert"] = np.zeros((nz + 2, ny + 2, nx + 2))
    rng = np.random.default_rng(seed)
    u = np.zeros((nz + 2, ny + 2, nx + 2, 3))
    u[1:-1, 1:-1, 1:-2, 0] = rng.standard_normal((nz, ny, nx - 1))
    u[1:-1, 1:-2, 1:-1, 1] = rng.standard_normal((nz, ny - 1, nx))
    u[1:-2, 1:-1, 1:-1, 2] = rng.standard_normal((nz - 1, ny, nx))
    f["ucont"] = u
    return cases.Case(name="affine", nx=nx, ny=ny, nz=nz, per=(0, 0, 0), bctype=(0,) * 6, immersed=0, fields=f)


def sheared_case(nx, ny, nz, per, seed=0):
    """The affine map of affine_case on any periodicity, with a sphere in the middle and a
    random flux field that carries nothing through the walls."""
    M = np.array([[1.0, 0.35, -0.2], [0.15, 0.8, 0.1], [-0.25, 0.3, 1.2]])
    P = np.stack(np.meshgrid(np.arange(nx + 1) / nx, np.arange(ny + 1) / ny, np.arange(nz + 1) / nz,
                             indexing="ij"), -1).transpose(2, 1, 0, 3)
    f = cases.form_metrics(cases.dmda_coords(P @ M.T), per)
    centre = cases.cell_centres(cases.dmda_coords(P))
    nv = cases.classify_nvert(cases.interior_only(cases.inside_sphere(centre, (0.45, 0.55, 0.5), 0.2)))
    cases.periodic_fill(nv, per)
    f["nvert"] = nv
    u = np.zeros(nv.shape + (3,))
    u[1:-1, 1:-1, 1:-1] = np.random.default_rng(seed).standard_normal((nz, ny, nx, 3))
    for a in range(3):
        if not per[a]:
            np.moveaxis(u[..., a], 2 - a, 0)[-2] = 0.0
    cases.set_periodic_flux_ghosts(u, per)
    f["ucont"] = u
    return cases.Case(name=f"sheared{nx}x{ny}x{nz}per{''.join(map(str, per))}", nx=nx, ny=ny, nz=nz, per=per,
                      bctype=(0,) * 6, immersed=1, fields=f)


def _sphere_immersed0():
    c = cases.hill_case(24, 16, 16, h=0.3, sphere=(0.6, 0.75, 0.0, 0.3), seed=1)
    c.immersed = 0
    c.name += "-immersed0"
    return c


CASES = {
    "channel": lambda: cases.channel_case(16, 16, 12, beta=2.0, seed=0),
    "hill_sphere": lambda: cases.hill_case(24, 16, 16, h=0.3, sphere=(0.6, 0.75, 0.0, 0.3), seed=0),
    "hill_sphere_immersed0": _sphere_immersed0,
    "towers": lambda: cases.towers_case(48, 24, 24, ratio=1.05, rows=2, cols=2, radius_cells=3, seed=2),
    "affine": affine_case,
}
_cache = {}


def get_case(name):
    if name not in _cache:
        c = CASES[name]()
        _cache[name] = (c, O.Assembled(c, drop=False), O.reference_projection(c, rtol=1e-13))
    return _cache[name]


def handle_for(E, c, **kw):
    h = E.Handle(E.make_grid(c.nx, c.ny, c.nz, c.per, c.bctype, c.immersed), E.default_opts(**kw))
    h.set_geometry(c.fields)
    return h


def relL2(a, b, mask):
    return float(np.linalg.norm((a - b)[mask]) / np.linalg.norm(b[mask]))


@pytest.fixture(scope="module")
def E(torch_cuda):
    from vfs_v3p2_amd import engine

    engine.lib()
    return engine


# ------------------------------------------------------------------ operator

@pytest.mark.parametrize("name", list(CASES))
def test_stencil_bit_exact(E, name):
    c, A, _ = get_case(name)
    h = handle_for(E, c)
    vol, cs = h.export_stencil()
    h.close()
    np.testing.assert_array_equal(cs, A.cases)
    np.testing.assert_array_equal(vol, A.vol)


@pytest.mark.parametrize("name", list(CASES))
def test_apply_matches_oracle(E, name, torch_cuda):
    torch = torch_cuda
    c, A, _ = get_case(name)
    h = handle_for(E, c)
    rng = np.random.default_rng(11)
    phi = rng.standard_normal(c.shape)
    cases.periodic_fill(phi, c.per)
    y_ref = O.stencil_apply(A.g, A.vol, A.rowflag, phi)
    tol = 1e-13 * np.abs(A.vol).max() * np.abs(phi).max() * 19
    pd = torch.from_numpy(phi).cuda()
    y = torch.zeros_like(pd)
    h.apply(pd, y, drop_small=False)
    fl = A.fluid_cells
    np.testing.assert_allclose(y.cpu().numpy()[fl], y_ref[fl], rtol=0, atol=tol)
    # the assembled matrix with the |a| <= 1e-10 drop rule
    rp, col, val = O.assemble_csr(A.g, A.vol, A.rowflag, A.gid, A.n, drop=True)
    yd_ref = O.csr_matvec(rp, col, val, A.to_compact(phi))
    h.apply(pd, y, drop_small=True)
    np.testing.assert_allclose(y.cpu().numpy()[fl], yd_ref, rtol=0, atol=tol)
    h.close()


# ------------------------------------------------------- reference primitives

def _inside_mask(shape, seed):
    c = cases.hill_case(shape[2], shape[1], shape[0], h=0.3, sphere=None, seed=0)
    co = cases.dmda_coords(cases.make_nodes(shape[2], shape[1], shape[0], -3 + np.arange(shape[2] + 1) * 6 / shape[2],
                                            np.arange(shape[1] + 1) / shape[1],
                                            -2 + np.arange(shape[0] + 1) * 4 / shape[0], hill_h=0.3))
    ins = cases.inside_sphere(cases.cell_centres(co), (0.4, 0.7, 0.1), 0.5)
    rng = np.random.default_rng(seed)
    ins |= rng.random(ins.shape) < 0.03  # isolated speckles exercise the neighbour rules
    return cases.interior_only(ins), c


@pytest.mark.parametrize("bctype", [(0, 0, 1, 1, 0, 0), (1, 1, 1, 1, 1, 1)])
def test_classify_nvert_bit_exact(E, torch_cuda, bctype):
    torch = torch_cuda
    ins, c = _inside_mask((16, 12, 20), 3)
    nv = np.where(ins, 4.0, 0.0)
    g = E.make_grid(20, 12, 16, c.per, bctype)
    d = torch.from_numpy(nv.copy()).cuda()
    E.classify_nvert_device(g, d)
    O.nvert_classify(O.grid(nv.shape, c.per), bctype, nv)
    np.testing.assert_array_equal(d.cpu().numpy(), nv)


def test_reference_multigrid_primitives_bit_exact(E, torch_cuda):
    torch = torch_cuda
    ins, c = _inside_mask((16, 12, 20), 5)
    nvf = np.where(ins, 4.0, 0.0)
    gf = O.grid(nvf.shape, (0, 0, 0))
    O.nvert_classify(gf, c.bctype, nvf)
    g = E.make_grid(20, 12, 16, (0, 0, 0), c.bctype)
    gc = O.grid(E.coarse_dmda_shape(g), (0, 0, 0))
    nvc_ref = O.mg_nvert_restrict(gf, gc, nvf)
    T = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    nvc = torch.zeros(E.coarse_dmda_shape(g), dtype=torch.float64, device="cuda")
    E.mg_nvert_restrict_device(g, T(nvf), nvc)
    np.testing.assert_array_equal(nvc.cpu().numpy(), nvc_ref)
    rng = np.random.default_rng(2)
    xf = rng.standard_normal(nvf.shape)
    xc = rng.standard_normal(nvc_ref.shape)
    fc = torch.zeros_like(nvc)
    E.mg_restrict_device(g, T(nvf), T(nvc_ref), T(xf), fc)
    np.testing.assert_array_equal(fc.cpu().numpy(), O.mg_restrict(gf, gc, nvf, nvc_ref, xf))
    ff = torch.zeros(nvf.shape, dtype=torch.float64, device="cuda")
    E.mg_prolong_device(g, T(nvf), T(nvc_ref), T(xc), ff)
    np.testing.assert_array_equal(ff.cpu().numpy(), O.mg_prolong(gf, gc, nvf, nvc_ref, xc))


# --------------------------------------------------------- full projection

@pytest.mark.parametrize("precision", [1, 0])
@pytest.mark.parametrize("name", list(CASES))
def test_projection_parity(E, name, precision):
    c, A, ref = get_case(name)
    print(f"case {name} {c.nx}x{c.ny}x{c.nz} precision {precision}", flush=True)
    user = E.UserCtx(c, E.default_opts(precision=precision, rtol=1e-12))
    st = E.Flow_Solver_pressure_step(user, strict=True)
    fl = A.fluid_cells
    phi = user.Phi.cpu().numpy()
    assert relL2(phi, ref["phi"], fl) <= PHI_TOL
    assert relL2(user.P.cpu().numpy(), ref["p"], fl) <= PHI_TOL
    assert st.max_div <= DIV_TOL and ref["maxdiv"] <= DIV_TOL
    # projection and Contra2Cart of the engine's own phi, by the oracle
    u = np.ascontiguousarray(c.fields["ucont"].copy())
    vf = O.volume_flux(A.g, c.immersed, u, c.fields)
    np.testing.assert_allclose(st.ibm_flux, vf[:4], rtol=1e-12, atol=1e-15)
    O.projection(A.g, c.fields, np.ascontiguousarray(phi), u, c.dt, c.st, c.coeff)
    ucat = np.zeros_like(u)
    O.contra2cart(A.g, c.bctype, c.fields, u, ucat)
    ug = user.Ucont.cpu().numpy()
    np.testing.assert_allclose(ug, u, rtol=0, atol=1e-13 * np.abs(u).max())
    np.testing.assert_allclose(user.Ucat.cpu().numpy(), ucat, rtol=0, atol=1e-13 * np.abs(ucat).max())
    md = O.divergence(A.g, ug, np.ascontiguousarray(c.fields["aj"]), A.nvert)
    assert abs(md - st.max_div) <= 1e-12 * max(md, 1e-300) + 1e-20
    assert abs(E.Divergence(user) - st.max_div) <= 1e-15
    user.handle.close()


@pytest.mark.parametrize("precision", [1, 0])
@pytest.mark.parametrize("name", list(CASES))
def test_fused_launches_are_bit_identical(E, torch_cuda, name, precision):
    """The fused launches (option `fused`) give the same bits as the separate ones:
    bit 0, the FP32 V-cycle's bottom (the last point level of at most 1024 cells and
    the dense solve in one workgroup); bit 1, the finest level's f D^-1 stored by
    the writers of the V-cycle input and read by its fused first Chebyshev steps.
    phi, P, Ucont, Ucat and the iteration count are compared for every combination
    against fused=0.  The hill cases (periodic in i and k) put the tail on level 1
    (12x8x8 above a 6x4x4 dense level), the affine box on the finest level itself
    (10x9x8, so its final x is the V-cycle's output); the other cases end in y-line
    or larger levels and must not take it, nor does the FP64 hierarchy."""
    torch = torch_cuda
    c, _, _ = get_case(name)
    tail_expected = precision == 1 and name in ("hill_sphere", "hill_sphere_immersed0", "affine")
    outs = {}
    for fused in (0, 1, 2, 3):
        h = handle_for(E, c, rtol=1e-12, precision=precision, fused=fused)
        desc = h.describe()
        print(f"case {name} precision {precision} fused {fused}:\n{desc}", flush=True)
        assert ("coarse tail" in desc) == (tail_expected and (fused & 1) == 1)
        u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
        phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
        p = torch.zeros_like(phi)
        ucat = torch.zeros(c.shape + (3,), dtype=torch.float64, device="cuda")
        st = h.project(u, phi, p, ucat, c.dt, c.st, c.coeff, strict=True)
        outs[fused] = (st.iterations, phi.cpu().numpy(), p.cpu().numpy(), u.cpu().numpy(), ucat.cpu().numpy())
        h.close()
    for fused in (1, 2, 3):
        assert outs[fused][0] == outs[0][0]
        for x, y in zip(outs[fused][1:], outs[0][1:]):
            np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("dims", [(32, 2, 16), (24, 20, 2)])
def test_coarse_tail_thin_axes(E, torch_cuda, dims):
    """The coarse tail's restriction when an axis of the tail level has fewer than 3
    cells and is not coarsened: j kept (32x2x16 -> 16x2x8, pairs in i and k) and k
    kept (24x20x2 -> 12x10x2, the per-child sum of the general restriction), on the
    finest level of a sheared non-periodic box, bit for bit against one launch per
    step (point smoothing forced, so the finest level is the tail level)."""
    torch = torch_cuda
    c = affine_case(*dims, seed=5)
    outs = []
    for fused in (3, 2):
        h = handle_for(E, c, rtol=1e-12, fused=fused, smoother=1)
        desc = h.describe()
        print(f"dims {dims} fused {fused}:\n{desc}", flush=True)
        assert ("coarse tail" in desc) == (fused == 3)
        u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
        phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
        p = torch.zeros_like(phi)
        ucat = torch.zeros(c.shape + (3,), dtype=torch.float64, device="cuda")
        st = h.project(u, phi, p, ucat, c.dt, c.st, c.coeff, strict=True)
        outs.append((st.iterations, phi.cpu().numpy(), u.cpu().numpy()))
        h.close()
    assert outs[0][0] == outs[1][0]
    for a, b in zip(outs[0][1:], outs[1][1:]):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("degree", [1, 2, 4])
def test_coarse_tail_chebyshev_degrees(E, torch_cuda, degree):
    """The coarse tail's step sequence for other Chebyshev degrees: one step from zero
    (degree 1, no fused pair), the fused pair alone (degree 2) and the fused pair
    with two further steps (degree 4), bit for bit against one launch per step
    (fused bit 0 clear)."""
    torch = torch_cuda
    c, _, _ = get_case("hill_sphere")
    outs = []
    for tail in (1, 0):
        h = handle_for(E, c, rtol=1e-12, cheb_degree=degree, fused=3 if tail else 2)
        assert ("coarse tail" in h.describe()) == (tail == 1)
        u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
        phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
        p = torch.zeros_like(phi)
        ucat = torch.zeros(c.shape + (3,), dtype=torch.float64, device="cuda")
        st = h.project(u, phi, p, ucat, c.dt, c.st, c.coeff, strict=True)
        print(f"degree {degree} coarse tail {tail}: {st.iterations} iterations", flush=True)
        outs.append((st.iterations, phi.cpu().numpy(), u.cpu().numpy()))
        h.close()
    assert outs[0][0] == outs[1][0]
    for a, b in zip(outs[0][1:], outs[1][1:]):
        np.testing.assert_array_equal(a, b)


def test_drop_rule_solve(E):
    """drop_small=1 solves the assembled HYPRE matrix (|a| <= 1e-10 dropped)."""
    c = cases.hill_case(16, 10, 12, h=0.3, sphere=(0.5, 0.8, 0.0, 0.4), seed=6)
    A = O.Assembled(c, drop=True)
    ref = O.reference_projection(c, rtol=1e-12, drop=True)
    user = E.UserCtx(c, E.default_opts(precision=0, rtol=1e-11, drop_small=1))
    st = E.Flow_Solver_pressure_step(user, strict=True)
    assert relL2(user.Phi.cpu().numpy(), ref["phi"], A.fluid_cells) <= PHI_TOL
    assert st.max_div <= DIV_TOL
    user.handle.close()


def test_deterministic_across_handles_and_calls(E, torch_cuda):
    torch = torch_cuda
    c, A, _ = get_case("hill_sphere")
    outs = []
    for _ in range(2):
        h = handle_for(E, c)
        for _ in range(2):
            u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
            phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
            p = torch.zeros_like(phi)
            ucat = torch.zeros(c.shape + (3,), dtype=torch.float64, device="cuda")
            h.project(u, phi, p, ucat, c.dt, c.st, c.coeff, strict=True)
            outs.append((phi.cpu().numpy(), u.cpu().numpy(), ucat.cpu().numpy()))
        h.close()
    for o in outs[1:]:
        for a, b in zip(o, outs[0]):
            np.testing.assert_array_equal(a, b)


def test_warm_start_from_previous_phi(E, torch_cuda):
    """zero_guess=0 starts from the Phi passed in, as the reference's persistent
    HYPRE vector does: the next step's solution is the same, in fewer iterations."""
    torch = torch_cuda
    c, A, _ = get_case("hill_sphere")
    h = handle_for(E, c, rtol=1e-12)
    u0 = np.ascontiguousarray(c.fields["ucont"])
    u1 = u0 * (1.0 + 0.01 * np.random.default_rng(4).standard_normal(u0.shape))
    cases.set_periodic_flux_ghosts(u1, c.per)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
    h.poisson_solve(dev(u0), phi, c.dt, c.st, c.coeff, strict=True)
    phi_cold = torch.zeros_like(phi)
    cold = h.poisson_solve(dev(u1), phi_cold, c.dt, c.st, c.coeff, strict=True)
    h.set_opts(zero_guess=0)
    warm = h.poisson_solve(dev(u1), phi, c.dt, c.st, c.coeff, strict=True)
    assert warm.iterations < cold.iterations
    assert relL2(phi.cpu().numpy(), phi_cold.cpu().numpy(), A.fluid_cells) <= PHI_TOL
    h.close()


def test_host_array_entry_matches_device(E, torch_cuda):
    torch = torch_cuda
    c, A, _ = get_case("towers")
    h = handle_for(E, c)
    u = np.ascontiguousarray(c.fields["ucont"].copy())
    phi = np.zeros(c.shape)
    p = np.zeros(c.shape)
    ucat = np.zeros(c.shape + (3,))
    h.project_host(u, phi, p, ucat, c.dt, c.st, c.coeff)
    ud = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
    phid = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
    pd = torch.zeros_like(phid)
    ucatd = torch.zeros(c.shape + (3,), dtype=torch.float64, device="cuda")
    h.project(ud, phid, pd, ucatd, c.dt, c.st, c.coeff)
    for a, b in ((u, ud), (phi, phid), (p, pd), (ucat, ucatd)):
        np.testing.assert_array_equal(a, b.cpu().numpy())
    h.close()


def test_error_behaviour(E, torch_cuda):
    torch = torch_cuda
    with pytest.raises(E.VfsPPError) as ei:
        E.Handle(E.make_grid(1, 8, 8))
    assert ei.value.code == E.VFS_PP_EINVAL
    c, A, _ = get_case("channel")
    h = E.Handle(E.make_grid(c.nx, c.ny, c.nz, c.per, c.bctype, c.immersed))
    u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
    phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
    with pytest.raises(E.VfsPPError) as ei:
        h.poisson_solve(u, phi, c.dt, c.st, c.coeff)
    assert ei.value.code == E.VFS_PP_ESTATE
    h.set_geometry(c.fields)
    bad = u.clone()
    bad[3, 4, 5, 0] = float("nan")
    with pytest.raises(E.VfsPPError) as ei:
        h.poisson_solve(bad, phi, c.dt, c.st, c.coeff)
    assert ei.value.code == E.VFS_PP_ENONFINITE
    with pytest.raises(ValueError):
        h.poisson_solve(u[:-1].contiguous(), phi, c.dt, c.st, c.coeff)
    # an iteration cap too small to converge is reported, not silent
    h.set_opts(max_iters=1, rtol=1e-14)
    with pytest.raises(E.VfsPPError) as ei:
        h.poisson_solve(u.clone(), phi, c.dt, c.st, c.coeff, strict=True)
    assert ei.value.code == E.VFS_PP_ENOCONV
    st = h.poisson_solve(u.clone(), phi, c.dt, c.st, c.coeff)
    assert st.converged == 0 and st.iterations == 1
    h.close()


# --------------------------------------------- the 192x96x128 terrain system

@pytest.fixture(scope="module")
def big():
    c = cases.hill_case(192, 96, 128, h=0.3, s=0.5, sphere=(0.6, 0.75, 0.0, 0.15), seed=0)
    return c, O.Assembled(c, drop=False)


@pytest.fixture(scope="module")
def big_runs(E, big, torch_cuda):
    c, A = big
    out = {}
    for prec in (1, 0):
        print(f"hill 192x96x128 + sphere, precision {prec}", flush=True)
        user = E.UserCtx(c, E.default_opts(precision=prec, rtol=2e-11))
        st = E.Flow_Solver_pressure_step(user, strict=True)
        out[prec] = (st, user.Phi.cpu().numpy(), user.Ucont.cpu().numpy(), user.Ucat.cpu().numpy())
        user.handle.close()
    return out


def test_big_divergence_free_both_forms(big, big_runs):
    c, A = big
    for prec in (1, 0):
        st, phi, u, _ = big_runs[prec]
        assert st.converged and st.max_div <= DIV_TOL
        md = O.divergence(A.g, u, np.ascontiguousarray(c.fields["aj"]), A.nvert)
        assert md <= DIV_TOL and abs(md - st.max_div) <= 1e-12 * md + 1e-20
        # null space removed: fluid mean of phi is zero
        lt = (A.nvert < 0.1)[1:-1, 1:-1, 1:-1]
        assert abs(phi[1:-1, 1:-1, 1:-1][lt].mean()) <= 1e-12 * np.abs(phi).max()


def test_big_mixed_equals_fp64(big, big_runs):
    c, A = big
    assert relL2(big_runs[1][1], big_runs[0][1], A.fluid_cells) <= PHI_TOL


def test_big_against_cpu_multigrid_oracle(big, big_runs):
    """The oracle's FP64 multigrid FGMRES on the CPU reaches the same phi."""
    c, A = big
    mg = O.CpuMG(A)
    r = O.cpu_projection(c, A, mg, rtol=1e-12)
    mg.close()
    assert relL2(big_runs[0][1], r["phi"], A.fluid_cells) <= PHI_TOL
    assert relL2(big_runs[1][1], r["phi"], A.fluid_cells) <= PHI_TOL


def test_big_projection_consistent_with_oracle(big, big_runs):
    c, A = big
    st, phi, ug, ucg = big_runs[1]
    u = np.ascontiguousarray(c.fields["ucont"].copy())
    O.volume_flux(A.g, c.immersed, u, c.fields)
    O.projection(A.g, c.fields, np.ascontiguousarray(phi), u, c.dt, c.st, c.coeff)
    np.testing.assert_allclose(ug, u, rtol=0, atol=1e-13 * np.abs(u).max())
    ucat = np.zeros_like(u)
    O.contra2cart(A.g, c.bctype, c.fields, u, ucat)
    np.testing.assert_allclose(ucg, ucat, rtol=0, atol=1e-13 * np.abs(ucat).max())


def test_divergence_rule_drives_the_solve(E, torch_cuda):
    """With div_tol set the solve goes on until the projected field meets it,
    whatever rtol says: max|aj div u| after projection = dt/coeff max|aj (b - A phi)|."""
    torch = torch_cuda
    c = cases.channel_case(24, 32, 16, beta=3.0, seed=3)
    out = {}
    for tag, dtol in (("loose", 0.0), ("ruled", 1e-8)):
        h = handle_for(E, c, rtol=1e-6, div_tol=dtol)
        u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
        phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
        p = torch.zeros_like(phi)
        ucat = torch.zeros(c.shape + (3,), dtype=torch.float64, device="cuda")
        out[tag] = h.project(u, phi, p, ucat, c.dt, c.st, c.coeff)
        h.close()
    assert out["loose"].max_div > 1e-8  # rtol alone does not get there on this grid
    assert out["ruled"].converged and out["ruled"].max_div <= 1e-8
    assert out["ruled"].iterations > out["loose"].iterations



@pytest.mark.parametrize("orthog", [1, 2])
@pytest.mark.parametrize("precision", [1, 0])
@pytest.mark.parametrize("name", ["hill_sphere", "towers", "affine"])
def test_orthogonalisation_variants(E, torch_cuda, name, precision, orthog):
    """Every Gram-Schmidt variant reaches the oracle's phi and a divergence-free
    field, in about the iterations of the default three-pass CGS2."""
    torch = torch_cuda
    c, A, ref = get_case(name)
    print(f"orthog {orthog} case {name} precision {precision}", flush=True)
    its = {}
    for o in (0, orthog):
        h = handle_for(E, c, precision=precision, rtol=1e-12, orthog=o)
        u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
        phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
        p = torch.zeros_like(phi)
        ucat = torch.zeros(c.shape + (3,), dtype=torch.float64, device="cuda")
        st = h.project(u, phi, p, ucat, c.dt, c.st, c.coeff, strict=True)
        h.close()
        its[o] = st.iterations
        assert relL2(phi.cpu().numpy(), ref["phi"], A.fluid_cells) <= PHI_TOL
        assert st.max_div <= DIV_TOL and st.rel_residual <= 1e-12
    assert abs(its[orthog] - its[0]) <= 1



@pytest.mark.parametrize("precision", [1, 0])
@pytest.mark.parametrize("dt,st,coeff", [(0.01, 0.5, 1.5), (0.01, 1.0, 1.5)])
def test_projection_parity_time_factors(E, dt, st, coeff, precision):
    """coeff = 1.5 is time_coeff() under rans after the first step (poisson.c:22-30);
    st (user->st) and dt enter the RHS as st coeff/dt (poisson_hypre.c:376) and the
    projection as dt st/coeff (poisson.c:2263).  The engine matches the oracle with
    these values.  Only st = 1 makes the projected field divergence-free (the RHS
    and the projection both scale by st), so max|div u| is checked there."""
    import dataclasses

    c0, A, _ = get_case("hill_sphere")
    c = dataclasses.replace(c0, dt=dt, st=st, coeff=coeff)
    ref = O.reference_projection(c, rtol=1e-13)
    print(f"hill_sphere dt {dt} st {st} coeff {coeff} precision {precision}", flush=True)
    user = E.UserCtx(c, E.default_opts(precision=precision, rtol=1e-12))
    stt = E.Flow_Solver_pressure_step(user, strict=True)
    fl = A.fluid_cells
    assert relL2(user.Phi.cpu().numpy(), ref["phi"], fl) <= PHI_TOL
    assert relL2(user.P.cpu().numpy(), ref["p"], fl) <= PHI_TOL
    # the oracle's projection of the engine's own phi (the engine folds dt st/coeff
    # into one factor, the reference applies them in turn: rounding-level agreement)
    u = np.ascontiguousarray(c.fields["ucont"].copy())
    O.volume_flux(A.g, c.immersed, u, c.fields)
    O.projection(A.g, c.fields, np.ascontiguousarray(user.Phi.cpu().numpy()), u, dt, st, coeff)
    np.testing.assert_allclose(user.Ucont.cpu().numpy(), u, rtol=0, atol=1e-13 * np.abs(u).max())
    ucat = np.zeros_like(u)
    O.contra2cart(A.g, c.bctype, c.fields, u, ucat)
    np.testing.assert_allclose(user.Ucat.cpu().numpy(), ucat, rtol=0, atol=1e-13 * np.abs(ucat).max())
    md = O.divergence(A.g, user.Ucont.cpu().numpy(), np.ascontiguousarray(c.fields["aj"]), A.nvert)
    assert abs(md - stt.max_div) <= 1e-12 * max(md, 1e-300) + 1e-20
    if st == 1.0:
        assert stt.max_div <= DIV_TOL and ref["maxdiv"] <= DIV_TOL
    else:
        assert stt.max_div > 1e-3 and abs(stt.max_div - ref["maxdiv"]) <= 1e-8 * ref["maxdiv"]
    user.handle.close()


def test_immersed_3_is_the_four_argument_volume_flux(E, torch_cuda):
    """immersed = 3 takes VolumeFlux(user, Ucont, ..) and zeroes the corrected faces
    like immersed = 0 (poisson_hypre.c:667, poisson.c:2728): identical results."""
    torch = torch_cuda
    outs = []
    for imm in (0, 3):
        c = _sphere_immersed0()
        h = E.Handle(E.make_grid(c.nx, c.ny, c.nz, c.per, c.bctype, imm), E.default_opts(rtol=1e-12))
        h.set_geometry(c.fields)
        u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
        phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
        p = torch.zeros_like(phi)
        ucat = torch.zeros(c.shape + (3,), dtype=torch.float64, device="cuda")
        st = h.project(u, phi, p, ucat, c.dt, c.st, c.coeff, strict=True)
        outs.append((phi.cpu().numpy(), u.cpu().numpy(), list(st.ibm_flux)))
        h.close()
    for a, b in zip(outs[0], outs[1]):
        np.testing.assert_array_equal(a, b)


def test_set_opts_after_a_failed_set_up(E):
    """A set-up that fails after the Krylov storage was sized (here: a coarse_max
    above the 1024-cell direct-solve limit leaves a 1728-cell coarsest level) still
    fixes precision and restart; hierarchy options may change, and the next set-up
    succeeds."""
    c = cases.channel_case(12, 12, 12, beta=2.0, seed=0)
    h = E.Handle(E.make_grid(c.nx, c.ny, c.nz, c.per, c.bctype, c.immersed), E.default_opts(coarse_max=2000))
    with pytest.raises(E.VfsPPError) as ei:
        h.set_geometry(c.fields)
    assert ei.value.code == E.VFS_PP_EINVAL
    for kw in ({"precision": 0}, {"restart": 12}):
        o = E.default_opts(coarse_max=2000, **kw)
        assert E.lib().vfs_pp_set_opts(h._h, E.C.byref(o)) == E.VFS_PP_ESTATE
    h.set_opts(coarse_max=512)
    h.set_geometry(c.fields)
    h.close()


def test_kernel_timer_ids(E, torch_cuda):
    """vfs_pp_time_kernel: every id times its kernel and states its algorithmic
    bytes (point levels: sweep 31 B/cell in FP32, streaming floor 35); a y-line
    finest level has no point-sweep streaming floor (EINVAL) and prices its fused
    residual + line step at 40 B/cell (records 24, x, previous x, f and the x it writes)."""
    c = get_case("hill_sphere")[0]
    h = handle_for(E, c, precision=1, smoother=1)
    n = c.nx * c.ny * c.nz
    print(f"time_kernel ids on {c.nx}x{c.ny}x{c.nz}", flush=True)
    for kid in (0, 1, 2, 3, 4, 6, 7, 8):
        ms, by = h.time_kernel(kid, 3)
        assert ms > 0 and by > 0, kid
    assert h.time_kernel(1, 3)[1] == 31 * n and h.time_kernel(8, 3)[1] == 35 * n
    h.close()
    ch = cases.channel_case(16, 64, 12, beta=3.0, seed=2)
    h = handle_for(E, ch, precision=1, smoother=2)
    assert h.time_kernel(1, 3)[1] == 40 * ch.nx * ch.ny * ch.nz
    with pytest.raises(E.VfsPPError) as ei:
        h.time_kernel(8, 3)
    assert ei.value.code == E.VFS_PP_EINVAL
    h.close()


@pytest.mark.parametrize("precision", [1, 0])
@pytest.mark.parametrize("ny", [136, 300])
def test_y_line_layouts_against_the_oracle(E, torch_cuda, precision, ny):
    """Every y-line level through the line kernels that its length selects: lines
    of up to 256 rows take the segmented, fused step (FP32: 16 segments of up to
    16 rows; FP64: 32 of up to 8), longer ones the residual kernel and one thread
    per line; nx = 20 leaves partial blocks.  Single-case and batched solves agree;
    the oracle's Divergence of the projected Ucont meets 1e-8 and the oracle's
    Projection of the engine's phi reproduces that Ucont; at ny = 136, where the
    CPU multigrid port converges, phi matches its solve."""
    torch = torch_cuda
    c = cases.channel_case(20, ny, 6, beta=2.5, seed=4)
    print(f"y-line layouts: channel 20x{ny}x6, precision {precision}", flush=True)
    A = O.Assembled(c, drop=False)
    outs = []
    for batched in (False, True):
        h = handle_for(E, c, precision=precision, smoother=2, rtol=1e-12)
        u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
        phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
        p = torch.zeros_like(phi)
        ucat = torch.zeros(c.shape + (3,), dtype=torch.float64, device="cuda")
        if batched:
            B = E.Batch([h])
            st = B.project([u], [phi], [p], [ucat], [c.dt], [c.st], [c.coeff], strict=True)[0]
            B.close()
        else:
            st = h.project(u, phi, p, ucat, c.dt, c.st, c.coeff, strict=True)
        assert "y-line" in h.describe()
        h.close()
        assert st.converged and st.max_div <= 1e-8
        outs.append((phi.cpu().numpy(), u.cpu().numpy()))
    assert relL2(outs[1][0], outs[0][0], A.fluid_cells) <= 1e-9
    phi, ug = outs[0]
    assert O.divergence(A.g, ug, np.ascontiguousarray(c.fields["aj"]), A.nvert) <= 1e-8
    u = np.ascontiguousarray(c.fields["ucont"].copy())
    O.volume_flux(A.g, c.immersed, u, c.fields)
    O.projection(A.g, c.fields, np.ascontiguousarray(phi), u, c.dt, c.st, c.coeff)
    np.testing.assert_allclose(ug, u, rtol=0, atol=1e-13 * np.abs(u).max())
    if ny == 136:
        mg = O.CpuMG(A)
        r = O.cpu_projection(c, A, mg, rtol=1e-12)
        mg.close()
        assert relL2(phi, r["phi"], A.fluid_cells) <= 1e-8


@pytest.mark.parametrize("dims", [(7, 64, 5), (21, 65, 3), (9, 129, 7), (17, 256, 3), (96, 33, 90), (128, 65, 67),
                                  (70, 130, 66), (130, 131, 127), (3, 40, 5), (130, 193, 128),
                                  (91, 225, 91)])
def test_y_line_block_layouts(E, torch_cuda, dims):
    """Every block layout of the segmented y-line step (line_layout: chosen by line
    length and line count, differently in FP32 and FP64), at odd sizes that leave
    partial blocks, short last segments and, where the grid holds it, a sphere whose
    rows take the decoded form.  The mixed and the FP64 solve meet rtol 1e-12, so their
    phi agree far below 1e-9, and a wrong line solve would not converge alike: the
    iteration counts differ by at most one."""
    torch = torch_cuda
    nx, ny, nz = dims
    c = (cases.hill_case(nx, ny, nz, h=0.3, beta=2.0, sphere=(0.6, 0.9, 0.0, 0.3), seed=6) if nx * nz > 4000
         else cases.channel_case(nx, ny, nz, beta=2.5, seed=6))
    print(f"y-line block layouts: {c.name}", flush=True)
    fluid = c.fields["nvert"][1:-1, 1:-1, 1:-1] < 0.1
    outs = []
    for precision in (1, 0):
        h = handle_for(E, c, precision=precision, smoother=2, rtol=1e-12)
        u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
        phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
        p = torch.zeros_like(phi)
        ucat = torch.zeros(c.shape + (3,), dtype=torch.float64, device="cuda")
        st = h.project(u, phi, p, ucat, c.dt, c.st, c.coeff, strict=True)
        h.close()
        assert st.max_div <= 1e-8
        outs.append((phi.cpu().numpy()[1:-1, 1:-1, 1:-1][fluid], st.iterations))
    (a, ia), (b, ib) = outs
    assert np.linalg.norm(a - b) <= 1e-9 * np.linalg.norm(b)
    assert abs(ia - ib) <= 1


@pytest.mark.parametrize("precision", [1, 0])
def test_iteration_queued_ahead(E, torch_cuda, precision):
    """The next V-cycle is queued before this iteration's scalars are read, and a zero
    start's first iteration before ||b|| is: a zero right-hand side, every iteration
    limit and loose and tight tolerances count iterations and V-cycles as if each were
    waited for.  (Results with a V-cycle queued in vain: test_vcycle_queued_in_vain.)"""
    torch = torch_cuda
    c = get_case("hill_sphere")[0]

    def solve(u, **kw):
        h = handle_for(E, c, precision=precision, **kw)
        phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
        st = h.poisson_solve(u, phi, c.dt, c.st, c.coeff)
        h.close()
        return st, phi.cpu().numpy()

    u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
    st, phi = solve(torch.zeros_like(u))
    assert st.converged and st.iterations == 0 and st.vcycles == 0 and st.rel_residual == 0.0 and not phi.any()
    for limit in (0, 1, 2, 5):
        st, phi = solve(u.clone(), max_iters=limit, rtol=1e-13, div_tol=0.0)
        assert not st.converged and st.iterations == limit and st.vcycles == limit and st.bnorm > 0.0
    last = 0
    for rtol in (0.5, 1e-2, 1e-5, 1e-9, 1e-12):
        st, _ = solve(u.clone(), rtol=rtol, div_tol=0.0)
        assert st.converged and st.rel_residual <= rtol and st.vcycles == st.iterations >= last
        last = st.iterations
    bad = u.clone()
    bad[3, 3, 3, 0] = float("nan")
    with pytest.raises(E.VfsPPError) as ei:
        solve(bad)
    assert ei.value.code == E.VFS_PP_ENONFINITE


# a V-cycle good enough for one iteration: many Chebyshev steps over nearly the whole spectrum
ONE_CYCLE = dict(cheb_degree=80, cheb_lo=0.003, coarse_max=100)


@pytest.mark.parametrize("precision", [1, 0])
@pytest.mark.parametrize("dims,kw,rtol", [((16, 12, 16), dict(smoother=1, **ONE_CYCLE), 5e-4),
                                          ((16, 12, 16), dict(smoother=2, **ONE_CYCLE), 5e-4),
                                          ((7, 6, 8), dict(coarse_max=512), 1e-5)])
def test_vcycle_queued_in_vain(E, torch_cuda, dims, kw, rtol, precision):
    """A solve that converges in its first iteration.  The second V-cycle is queued before
    that is known (always, at the first iteration of a zero start with rtol below 1e-3), unless
    max_iters = 1 says that there is none: the two give the same bits.  Systems: two levels
    with the point and with the y-line smoother, and a grid that is its own dense level,
    where the first basis vector cancels to rounding and the re-orthogonalisation discards
    the queued V-cycle.  A zero and a non-finite right-hand side leave queued
    V-cycles behind too: the next solve on the handle has the fresh handle's bits."""
    torch = torch_cuda
    nx, ny, nz = dims
    c = cases.hill_case(nx, ny, nz, h=0.1, beta=0.0, sphere=None, seed=2)
    print(f"V-cycle in vain: {c.name} {kw}, precision {precision}", flush=True)
    u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()

    def solve(h, ucont):
        phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
        st = h.poisson_solve(ucont, phi, c.dt, c.st, c.coeff)
        return st, phi.cpu().numpy()

    out = []
    for more in (dict(max_iters=1), {}):
        h = handle_for(E, c, precision=precision, rtol=rtol, div_tol=0.0, **kw, **more)
        out.append(solve(h, u.clone()))
        if more:
            h.close()
    (st1, phi1), (st, phi) = out
    assert st1.converged and st.converged and st1.iterations == st.iterations == st.vcycles == 1
    assert phi1.any() and np.array_equal(phi, phi1) and st.rel_residual == st1.rel_residual
    bad = u.clone()
    bad[2, 2, 2, 0] = float("nan")
    for rhs in (None, torch.zeros_like(u), bad):
        if rhs is bad:
            with pytest.raises(E.VfsPPError):
                solve(h, rhs)
        elif rhs is not None:
            assert solve(h, rhs)[0].iterations == 0
        assert np.array_equal(solve(h, u.clone())[1], phi)
    h.close()


@pytest.mark.parametrize("dims", [(3, 150, 150), (65, 34, 33), (127, 23, 25), (129, 33, 17), (130, 256, 3),
                                  (259, 191, 3), (40, 41, 39)])
def test_pair_walk(E, torch_cuda, dims):
    """The FP64 operator with two cells per thread (levels of 65536 cells on): rows shorter
    than a wave, odd rows whose last pair overlaps the one before, rows of one wave of
    pairs and one more, planes walked in slabs with a short last one, and one grid below
    the bound.  The converged Phi has to satisfy the system in the coefficient form, which
    shares none of that code: |b - A Phi| <= 1e-11 |b| from a true residual of 1e-12 |b|,
    with the rounding of a 19-term row on top (the two forms' rows differ by at most
    38 eps |A| |Phi|, far below 1e-11 |b| at these sizes)."""
    nx, ny, nz = dims
    _pair_walk(E, torch_cuda,
               cases.hill_case(nx, ny, nz, h=0.2, beta=1.5, sphere=(0.6, 0.9, 0.0, 0.25), seed=8)
               if nx > 100 and nz > 3 else cases.channel_case(nx, ny, nz, beta=1.5, seed=8))


@pytest.mark.parametrize("per", [(0, 0, 0), (1, 1, 1), (0, 1, 0), (0, 0, 1), (1, 1, 0)])
def test_pair_walk_on_other_topologies(E, torch_cuda, per):
    """test_pair_walk with walls in i and k and with periodic j, on a sheared grid with a
    sphere: the wrapped columns and rows of the pairs and the walls' one-sided rows."""
    _pair_walk(E, torch_cuda, sheared_case(65, 34, 33, per, seed=5))


def _pair_walk(E, torch, c):
    print(f"pair walk: {c.name}", flush=True)
    A = O.Assembled(c, drop=False)
    for precision in (0, 1):
        h = handle_for(E, c, precision=precision, rtol=1e-12, div_tol=0.0, max_iters=400)
        u = torch.from_numpy(np.ascontiguousarray(c.fields["ucont"])).cuda()
        phi = torch.zeros(c.shape, dtype=torch.float64, device="cuda")
        st = h.poisson_solve(u, phi, c.dt, c.st, c.coeff, strict=True)
        for ax, per in zip((2, 1, 0), c.per):  # the periodic images apply() reads
            if per:
                phi.select(ax, 0).copy_(phi.select(ax, -2))
                phi.select(ax, -1).copy_(phi.select(ax, 1))
        y = torch.zeros_like(phi)
        h.apply(phi, y)
        h.close()
        b = O.rhs(A.g, u.cpu().numpy(), A.nvert, c.dt, c.st, c.coeff)
        r = np.abs(y.cpu().numpy() - b)[A.fluid_cells]
        bn = np.linalg.norm(b[A.fluid_cells])
        assert st.converged and abs(st.bnorm - bn) <= 1e-12 * bn
        assert np.linalg.norm(r) <= 1e-11 * bn
