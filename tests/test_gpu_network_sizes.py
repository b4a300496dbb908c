"""The warm-start network on graphs of awkward sizes (fewer rows than a tile,
one more or less than a tile or a wave, a vertex with more neighbours than half
a wave has lanes): forward, loss and every gradient block against the oracle."""
import ctypes as C

import numpy as np
import pytest

from tests.conftest import relerr

pytestmark = pytest.mark.gpu


def _graph(n, rng):
    """A ring with random chords; vertex 0 is joined to (nearly) all others."""
    A = np.zeros((n, n), dtype=bool)
    i = np.arange(n)
    A[i, (i + 1) % n] = True
    A[0, 1:] = True
    A[rng.integers(0, n, 2 * n), rng.integers(0, n, 2 * n)] = True
    A |= A.T
    np.fill_diagonal(A, False)
    return np.concatenate([[0], np.cumsum(A.sum(1))]).astype(np.int64), np.nonzero(A)[1].astype(np.int32)


@pytest.mark.parametrize("n", [2, 31, 32, 33, 64, 65, 127, 300])
def test_forward_and_gradient(n):
    from m3tet_sph_amd import learned as L
    from m3tet_sph_amd.api import D, I32, I64, _p
    from oracle import gnn as OG
    rng = np.random.default_rng(n)
    ptr, col = _graph(n, rng)
    radius = rng.uniform(0.6, 0.9, n)
    net = L.WarmStartNet.__new__(L.WarmStartNet)
    net.n, net._h = n, C.c_void_p()
    d = L.GraphDesc()
    d.nvert, d.nnod, d.adj_ptr, d.adj_col, d.radius = n, n, _p(ptr, I64), _p(col, I32), _p(radius, D)
    d.r_in, d.r_out = 0.5, 1.0
    assert L.LIB.m3_gnn_create(C.byref(net._h), 0, C.byref(d)) == 0
    try:
        p = L.init_params(n) + 0.05 * rng.standard_normal(L.NPARAM).astype(np.float32)
        norm = np.concatenate([0.1 * rng.standard_normal(8), rng.uniform(0.5, 2, 12)]).astype(np.float32)
        X = rng.standard_normal((n, 8)).astype(np.float32)
        Y = rng.standard_normal((n, 4)).astype(np.float32)
        net.set_params(p, norm)
        pred, loss, grad = net.forward_backward(X, Y)
        l_ref, g_ref, y_ref = OG.loss_and_grad(X, Y, p, norm, ptr, col, exact=True)
        # FP32 sums of a few hundred terms; an activation on the edge of a BF16
        # rounding may fall the other way (2^-9 of one of 64 n values)
        assert relerr(pred, y_ref) < 1e-5 + 2e-3 / n
        assert abs(loss - l_ref) < 1e-4 * l_ref
        edges = [0, 512, 576] + [576 + k * 8256 + o for k in range(3) for o in (8192, 8256)] + [25600, L.NPARAM]
        for a, b in zip(edges, edges[1:]):
            assert relerr(grad[a:b], g_ref[a:b]) < 1e-4 + 2e-2 / n, (a, b)
    finally:
        net.close()
