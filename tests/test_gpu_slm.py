"""m3_advect3d_slm_p_sph (P2 semi-Lagrangian advection, the production
configuration of advect3d_slm_p_sph) against the restatement in
oracle/slm.py on the 3,840-tet shell, with a prescribed smooth flow and with
the velocity of a Stokes solve; identities on the c1 shell."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def log(*a):
    print("[gpu]", *a, flush=True)


def _flow(m):
    x, y, z = m.GCOORD.T
    return -y + 0.3 * x * z, x + 0.3 * y * z, -0.3 * (x * x + y * y)


def _field(m):
    th, ph, r = m.GCOORD_SPH.T
    return r * r + 0.3 * r * np.sin(2 * th) * np.cos(3 * ph)


def _compare(m, ctx, Ux, Uy, Uz, T, dt, monotonic, method_BT="PC2"):
    from oracle import slm as S
    Tg, info = ctx.advect3d_slm_p_sph(Ux, Uy, Uz, T, dt, monotonic=monotonic, method_BT=method_BT)
    To, d = S.advect3d_slm_p_sph(m, Ux, Uy, Uz, T, dt, monotonic=bool(monotonic), detail=True,
                                 method_BT=method_BT)
    scale = np.abs(T).max()
    diff = np.abs(Tg - To) / scale
    # departure points within 1e-8 of an element face may be assigned to
    # either element (and, across class frames, interpolated slightly
    # differently): those are checked against the bound of the clip only
    clear = d["m2"] > 1e-8
    log(f"nnod {m.nnod}: max |dT| {diff.max():.2e} ({diff[clear].max():.2e} away from faces, "
        f"{(~clear).sum()} near faces), shifted {info['nshift']}, unresolved {info['nunresolved']}")
    assert info["nunresolved"] == 0
    assert diff[clear].max() < 1e-9
    assert np.quantile(diff, 0.99) < 1e-9
    assert diff.max() < 1e-3
    return Tg


@pytest.fixture(scope="module")
def c0_ctx():
    from m3tet_sph_amd import api, mesh as M
    m = M.build_config("c0")
    ctx = api.StokesContext(m)
    yield m, ctx
    ctx.close()


@pytest.mark.parametrize("monotonic", [1, 0])
def test_prescribed_flow_matches_the_oracle(c0_ctx, monotonic):
    m, ctx = c0_ctx
    Ux, Uy, Uz = _flow(m)
    _compare(m, ctx, Ux, Uy, Uz, _field(m), 0.05, monotonic)


@pytest.mark.parametrize("monotonic", [1, 0])
def test_eu1_matches_the_oracle(c0_ctx, monotonic):
    """method_BT = 'EU1': the three arrays are (v_theta, v_phi, v_r), as the
    reference's backtrack_EU1 takes them."""
    m, ctx = c0_ctx
    th, ph, r = m.GCOORD_SPH.T
    vth, vph, vr = 0.5 * r * np.sin(ph), 0.8 * r + 0.2 * np.cos(th), 0.3 * np.cos(th) * np.sin(2 * ph)
    _compare(m, ctx, vth, vph, vr, _field(m), 0.05, monotonic, method_BT="EU1")


def test_eu1_radial_closed_form(c0_ctx):
    """EU1 with only v_r: a field linear in the radius lands on the
    back-tracked radius, clipped into the shell."""
    m, ctx = c0_ctx
    r = m.GCOORD_SPH[:, 2]
    z = np.zeros(m.nnod)
    T = 2.0 + 3.0 * r
    Tg, info = ctx.advect3d_slm_p_sph(z, z, np.full(m.nnod, 0.8), T, 0.05, method_BT="EU1")
    tol = 1e-12 * (r.max() - r.min())
    r_bt = np.clip(r - 0.05 * 0.8, r.min() + tol, r.max() - tol)
    assert np.abs(Tg - (2.0 + 3.0 * r_bt)).max() < 1e-9
    assert info["nshift"] == int((r - 0.05 * 0.8 <= r.min() + tol).sum())


def test_stokes_velocity_matches_the_oracle(c0_ctx):
    from m3tet_sph_amd import fields as F
    m, ctx = c0_ctx
    inp = F.make_inputs(m, visc_contrast=1e3)
    ctx.set_bc(inp["ifix"], inp["vfix"])
    U, P, info = ctx.flow3d(inp["Visc"], inp["Dens"], inp["phys"], rtol_Pat=1e-6)
    # rotated (theta, phi, r) components to Cartesian (make_rotation_matrix.m)
    th, ph, _ = m.GCOORD_SPH.T
    ct, st, cp, sp = np.cos(th), np.sin(th), np.cos(ph), np.sin(ph)
    a, b, c = U[0::3], U[1::3], U[2::3]
    Ux = cp * ct * a - sp * b + cp * st * c
    Uy = sp * ct * a + cp * b + sp * st * c
    Uz = -st * a + ct * c
    vmax = np.sqrt(Ux ** 2 + Uy ** 2 + Uz ** 2).max()
    dt = 0.5 * 0.05 / vmax
    _compare(m, ctx, Ux, Uy, Uz, _field(m), dt, 1)


def test_identities_on_c1():
    from m3tet_sph_amd import api, mesh as M
    import time
    m = M.build_config("c1")
    ctx = api.StokesContext(m)
    z = np.zeros(m.nnod)
    T = _field(m)
    T0, info = ctx.advect3d_slm_p_sph(z, z, z, T, 0.1)
    assert np.abs(T0 - T).max() < 1e-10 * np.abs(T).max()
    Ux, Uy, Uz = _flow(m)
    c = np.full(m.nnod, 0.25)
    assert np.array_equal(ctx.advect3d_slm_p_sph(Ux, Uy, Uz, c, 0.02)[0], c)
    t = time.perf_counter()
    Tn, info = ctx.advect3d_slm_p_sph(Ux, Uy, Uz, T, 0.02)
    dtw = time.perf_counter() - t
    assert Tn.min() >= T.min() and Tn.max() <= T.max() and info["nunresolved"] == 0
    log(f"c1 ({m.nnod} P2 nodes): {dtw * 1e3:.1f} ms per call including host copies, info {info}")
    with pytest.raises(api.M3Error):
        ctx.advect3d_slm_p_sph(Ux, Uy, Uz, T, 0.02, method_BT="RK4")
    bad = T.copy()
    bad[7] = np.nan
    with pytest.raises(api.M3Error):
        ctx.advect3d_slm_p_sph(Ux, Uy, Uz, bad, 0.02)
    ctx.close()


def test_another_mesh_in_the_same_context(tiny, c0):
    """The face table and the node frames belong to the mesh they were made for;
    a mesh that is refused leaves none to advect on."""
    import copy
    from m3tet_sph_amd import api
    ctx, fresh = api.StokesContext(tiny), api.StokesContext(c0)
    try:
        ctx.advect3d_slm_p_sph(*_flow(tiny), _field(tiny), 0.05)
        ctx._set_mesh(c0)
        got, _ = ctx.advect3d_slm_p_sph(*_flow(c0), _field(c0), 0.05)
        want, _ = fresh.advect3d_slm_p_sph(*_flow(c0), _field(c0), 0.05)
        assert np.array_equal(got, want)
        bad = copy.copy(c0)
        bad.levels = [copy.copy(L) for L in c0.levels]
        bad.levels[1].EL2NOD = c0.levels[1].EL2NOD + c0.levels[1].nnod
        with pytest.raises(api.M3Error, match="EL2NOD entry out of range"):
            ctx._set_mesh(bad)
        with pytest.raises(api.M3Error, match="before m3_set_mesh"):
            ctx.advect3d_slm_p_sph(*_flow(c0), _field(c0), 0.05)
        with pytest.raises(api.M3Error, match="before m3_set_mesh"):
            ctx.diffusion_mesh()
    finally:
        ctx.close()
        fresh.close()
