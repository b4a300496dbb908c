"""The sweeps of the multigrid levels against the stored operator: levels below
the window size limit (one slice per workgroup, its blocks dealt to waves), and
levels that are swept in windows, with a last window that is not full, with
windows split and given up, on generated shells and on the unstructured mesh file.  K x, the transfers and the
diagonal against SciPy products of m3_get_operator's matrix; one velocity solve
in both precisions against each other."""
import os

import numpy as np
import pytest

from tests.conftest import relerr

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(__file__), "golden", "EarthShell_n37k.mat")

# nodes of the finest level: 5,778 (a last slice of 18 rows), 92,178, 337,986
# (a last window of 66 rows), 289,174 of the file, 174,114 (a last window of 34 rows)
CASES = [dict(level=1, nlayer=2, nmg=2), dict(level=2, nlayer=1, nmg=3), dict(level=1, nlayer=2, nmg=4), None,
         dict(level=2, nlayer=2, nmg=3)]
WINDOWS = [0, 0, 661, 565, 341]

# The same with other windows (fewest rows, most entries of a window, of 64 rows,
# per row of the level; 0: the default).  Unforced, the windows of the 174,114 nodes gather 1,349
# entries on average and at most 1,705, their 64-row slices at most 447.  Levels
# of 174,114 and 23,058 nodes in windows, so that both ends of a transfer are in
# vector order; a few windows split; windows of 64 to 256 rows; of 64 rows alone;
# a slice that gathers too much, and windows that do in all (without a split and
# with one), so that a large level has none
FORCED = [(3, (2000, 0, 0, 0), lambda w: w == [341, 46, 0]),
          (3, (0, 1650, 0, 0), lambda w: 341 < w[0] < 400),
          (2, (1000, 600, 0, 100), lambda w: 2 * 46 < w[0] < 361),
          (2, (1000, 1, 0, 100), lambda w: w[0] == 361),
          (3, (0, 0, 300, 0), lambda w: w == [0, 0, 0]),
          (3, (0, 0, 0, 2), lambda w: w == [0, 0, 0]),
          (3, (0, 500, 0, 0), lambda w: w == [0, 0, 0])]


@pytest.mark.parametrize("k", range(len(CASES)), ids=["small", "direct", "windows", "file", "windows34"])
def test_level_operators(k):
    from m3tet_sph_amd import mesh as M
    m = M.build_from_file(GOLD, nmg=2, device=0) if CASES[k] is None else M.build_shell(**CASES[k], device=0)
    _check_levels(m, None, lambda w: w[0] == WINDOWS[k] and not any(w[1:]))


@pytest.mark.parametrize("nmg,rule,expect", FORCED, ids=["levels", "some_split", "split", "slices", "slice_too_large",
                                                                "too_many", "too_many_split"])
def test_level_operators_with_other_windows(nmg, rule, expect):
    from m3tet_sph_amd import mesh as M
    _check_levels(M.build_shell(level=2, nlayer=2, nmg=nmg, device=0), rule, expect)


def _check_levels(m, rule, expect):
    from m3tet_sph_amd import api, fields as F
    T = (m.r_surf - m.GCOORD_SPH[:, 2]) / (m.r_surf - m.r_cmb) + 0.03 * np.sin(7 * m.GCOORD[:, 0])
    Visc, Dens = F.material(T, 1e3)
    ifix, vfix = F.plate_bcs(m)
    ctx = api.StokesContext(m, sweep_windows=rule)
    try:
        st = ctx.stats()
        print("nodes", [L.nnod for L in m.levels], "windows", st["windows"], "entries", st["window_entries"])
        assert expect(st["windows"])
        ctx.set_bc(ifix, vfix)
        ctx.assemble(Visc, Dens, F.physics())
        ctx.restrict_stiffmat()
        ctx.cholesky_factorization()
        rng = np.random.default_rng(0)
        for l in range(m.nmg):
            K = api.get_operator(ctx, l)
            x = rng.standard_normal(K.shape[1])
            # sums of at most some 100 x 3 products in another order: n eps = 7e-14 at worst
            assert relerr(ctx.apply(0, l, x), K @ x) < 1e-13
            assert relerr(ctx.get_vector(2, l), K.diagonal()) < 1e-15
            assert abs(K - K.T).max() <= 1e-12 * abs(K).max()
        for l in range(m.nmg - 1):
            P = api.intermesh_transfer_matrix(m, l)
            mf, mc = ctx.get_vector(3, l), ctx.get_vector(3, l + 1)
            xc, xf = rng.standard_normal(P.shape[1]), rng.standard_normal(P.shape[0])
            assert relerr(ctx.apply(4, l, xc), mf * (P @ xc)) < 1e-13
            assert relerr(ctx.apply(5, l, xf), mc * (P.T @ xf)) < 1e-13
        b = ctx.get_vector(0) - ctx.get_vector(1)
        x64, n64, _ = ctx.mgpcg(b, tol=1e-9, is_abs_tol=False, itmax=60)
        x16, n16, _ = ctx.mgpcg(b, x=0.3 * x64, tol=1e-9, is_abs_tol=False, itmax=60, precision="mixed")
        K0, free = api.get_operator(ctx, 0), ctx.get_vector(3, 0)
        for x in (x64, x16):
            r = free * (b - K0 @ x)
            assert np.linalg.norm(r) < 2e-9 * np.linalg.norm(free * b)
        # both stop at the same residual; the operator's conditioning is below 1e5 here
        assert relerr(x16, x64) < 1e-4 and abs(n64 - n16) <= 3
    finally:
        ctx.close()


def _scattered(m):
    """The mesh with the Cartesian coordinates of its fine nodes outside the cones
    dealt out again: the elements there are formed from the spherical ones, so only
    the order of the nodes suffers (and the frames they are rotated to), and a
    window gathers thousands of entries."""
    import copy
    cone = np.concatenate([m.classes["in_cone_no_iso"], m.classes["in_cone_iso"]])
    free = np.ones(m.nnod, dtype=bool)
    free[: m.levels[-1].nnod] = False
    free[np.unique(m.levels[0].EL2NOD[cone])] = False
    i = np.nonzero(free)[0]
    out = copy.copy(m)
    out.GCOORD = m.GCOORD.copy()
    out.GCOORD[i] = m.GCOORD[np.random.default_rng(0).permutation(i)]
    return out


# the rule's own limits of a window (LDS of up to 82 KB in FP64), and as much as a
# workgroup can hold (163 KB); against the form that the rule chooses, no windows
@pytest.mark.parametrize("rule,entries", [((0, 0, 0, 100), (2300, 2900)), ((0, 6300, 6300, 100), (5000, 6300))],
                         ids=["split", "largest"])
def test_windows_that_gather_thousands(rule, entries):
    from m3tet_sph_amd import api, fields as F, mesh as M
    m = _scattered(M.build_shell(level=2, nlayer=2, nmg=3, device=0))
    T = (m.r_surf - m.GCOORD_SPH[:, 2]) / (m.r_surf - m.r_cmb)
    Visc, Dens = F.material(T, 1e2)
    x = np.random.default_rng(1).standard_normal(3 * m.nnod)
    got = []
    for r in (rule, None):
        ctx = api.StokesContext(m, sweep_windows=r)
        try:
            st = ctx.stats()
            print("windows", st["windows"], "entries", st["window_entries"], flush=True)
            if r is rule:
                assert st["windows"][0] > 341 and entries[0] < st["window_entries"][0] <= entries[1]
            else:
                assert st["windows"] == [0, 0, 0]
            ctx.set_bc(*F.plate_bcs(m))
            ctx.assemble(Visc, Dens, F.physics())
            ctx.restrict_stiffmat()
            ctx.cholesky_factorization()
            free = ctx.get_vector(3)
            b = free * ctx.apply(0, 0, free * x)
            got.append([b] + [ctx.mgpcg(b, tol=0.0, itmax=1, precision=p)[0] for p in ("fp64", "mixed")])
        finally:
            ctx.close()
    # one V-cycle and step: the sums of some 100 x 3 products in other orders, in
    # 64 and in 32 bits, through 14 sweeps
    for a, b, tol in zip(got[0], got[1], (1e-13, 1e-11, 1e-4)):
        assert relerr(a, b) < tol


def test_vectors_of_an_unfinished_mesh(tiny):
    """A mesh that is refused at its second level leaves the first one without
    its vectors: reading the diagonal of K raises."""
    import copy
    from m3tet_sph_amd import api
    ctx = api.StokesContext(tiny)
    try:
        bad = copy.copy(tiny)
        bad.levels = [copy.copy(L) for L in tiny.levels]
        bad.levels[1].EL2NOD = tiny.levels[1].EL2NOD + tiny.levels[1].nnod
        with pytest.raises(api.M3Error, match="EL2NOD entry out of range"):
            ctx._set_mesh(bad)
        with pytest.raises(api.M3Error):
            ctx.get_vector(2, 0)
    finally:
        ctx.close()
