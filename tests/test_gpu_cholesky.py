"""The coarsest level's factorisation and solve on root sizes that take each
form of the solves: the whole matrix as one block, some of the first
dissection levels merged, none merged."""
import os

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden", "EarthShell_n37k.mat")

# tiles of the coarsest level and launches of a solve's direction: 34 tiles as one
# block (four with no blocks merged), 73, 130 and 275 (five, six and seven), and
# the mesh file's 1,844, of which nothing is merged
CASES = [((1, 2, 2), 34, 1), ((1, 4, 4), 73, 2), ((2, 2, 2), 130, 3), ((2, 4, 3), 275, 6), (None, 1844, 10)]


@pytest.mark.parametrize("shape,tiles,heights", CASES, ids=[str(c[1]) for c in CASES])
def test_coarse_solve(shape, tiles, heights):
    from m3tet_sph_amd import api, fields as F, mesh as M
    m = M.build_shell(*shape, device=0) if shape else M.build_from_file(GOLD, nmg=2, device=0)
    T = (m.r_surf - m.GCOORD_SPH[:, 2]) / (m.r_surf - m.r_cmb) + 0.03 * np.sin(7 * m.GCOORD[:, 0])
    Visc, Dens = F.material(T, 1e3)
    ctx = api.StokesContext(m)
    try:
        ctx.set_bc(*F.plate_bcs(m))
        ctx.assemble(Visc, Dens, F.physics())
        ctx.restrict_stiffmat()
        ctx.cholesky_factorization()
        st = ctx.stats()
        assert st["chol_T"] == tiles and st["chol_heights"] == heights
        K = sp.csr_matrix(api.get_operator(ctx, m.nmg - 1))
        free = ctx.get_vector(3, m.nmg - 1) > 0
        b = np.random.default_rng(1).standard_normal(K.shape[1]) * free
        x = ctx.cholesky_solve(b)
        # backward error of a triangular factor's solve: below n eps in the
        # norm of |A| |x|, each of its n-term sums rounded once per term
        err = np.linalg.norm((b - K @ x)[free]) / np.linalg.norm((abs(K) @ abs(x))[free])
        print("coarse", st["chol_n"], st["chol_T"], st["chol_heights"], "err", err)
        assert err < st["chol_n"] * np.finfo(float).eps
    finally:
        ctx.close()
