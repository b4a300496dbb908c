"""The pressure iteration's fused vector steps against the same recurrence in
NumPy, on pressure meshes with a last slice that is not full, and with more
slices than workgroups.  Homogeneous velocities, so that U0 is zero."""
import numpy as np
import pytest

from tests.conftest import relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,nlayer,nmg", [(1, 2, 2), (2, 2, 2), (1, 4, 4)], ids=["small", "middle", "large"])
def test_pressure_iteration(level, nlayer, nmg):
    from m3tet_sph_amd import api, fields as F, mesh as M
    m = M.build_shell(level=level, nlayer=nlayer, nmg=nmg, device=0)
    T = (m.r_surf - m.GCOORD_SPH[:, 2]) / (m.r_surf - m.r_cmb) + 0.03 * np.sin(7 * m.GCOORD[:, 0])
    Visc, Dens = F.material(T, 10.0)
    ifix, vfix = F.plate_bcs(m)
    ctx = api.StokesContext(m)
    try:
        ctx.set_bc(ifix, 0.0 * vfix)
        ctx.assemble(Visc, Dens, F.physics())
        ctx.restrict_stiffmat()
        ctx.cholesky_factorization()
        free, Fb, L = ctx.get_vector(3), ctx.get_vector(0), ctx.get_vector(4)
        rng = np.random.default_rng(0)
        q, z = rng.standard_normal(m.nVnod), rng.standard_normal(3 * m.nnod)
        # the two products of a few hundred terms a row hold the same numbers
        assert abs(ctx.apply(2, 0, z) @ q - ctx.apply(1, 0, q) @ z) < 1e-12 * (
            np.linalg.norm(ctx.apply(1, 0, q)) * np.linalg.norm(z))
        opts = dict(rtol_Pat=1e-3, rtol_U=1e-8, itmax_U=80, itmin_Pat=4, itmax_Pat=4)
        _, P, info = ctx.patera(**opts)
        assert info["nitP"] == 4

        def solve(b):
            return ctx.mgpcg(b, tol=1e-11, is_abs_tol=False, itmax=80)[0]
        r = -ctx.apply(2, 0, solve(free * Fb))
        r -= r.mean()
        Pn, qn, rl, rd = np.zeros(m.nVnod), None, None, 0.0
        for it in range(4):
            p = r / L
            d = p + (r - ctx.apply(3, 0, p)) / L
            qn = d if it == 0 else d + ((r - rl) @ d) / rd * qn
            qn = qn - qn.mean()
            rd = r @ d
            Sq = ctx.apply(2, 0, solve(free * ctx.apply(1, 0, qn)))
            alpha = rd / (qn @ Sq)
            Pn, rl, r = Pn + alpha * qn, r, r - alpha * Sq
            r = r - r.mean()
        # the velocity solves' 1e-8 of the pressure residual, over four iterations
        # of a system whose conditioning is below 1e2
        assert relerr(P, Pn) < 1e-5
    finally:
        ctx.close()
