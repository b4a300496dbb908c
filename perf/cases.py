"""Performance cases: the work that a convection code has this framework do, called as such a code calls it.

A time loop on a spherical shell sets its mesh up once, then at every step makes the operators of the step's viscosity, solves the
Stokes problem (from nothing, from the previous steps, or from the learned start) and carries the temperature on.  The cases are these
calls on shells from a few thousand to two million elements, regular ones and the unstructured mesh file of the tests.  Every state
holds its own device context; what is made once per mesh (the mesh itself) is kept between states.

``exact`` gives the results in 64 bits from plain torch: its own element integration, dense factorisations for systems of up to
DENSE unknowns, its own conjugate gradients, its own network.
"""
import functools
import os

import numpy as np
import torch

from m3tet_sph_amd import api, learned, mesh as meshmod

HERE = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MESH_FILE = os.path.join(HERE, "tests", "golden", "EarthShell_n37k.mat")
NETWORK = os.path.join(HERE, "m3tet_sph_amd", "data", "warm_start_c1.npz")
PHYS = dict(g=-1.0, Bscale=1e5, Dens0=1.0, minVisc=None, maxVisc=None)
DENSE = 20000       # unknowns up to which exact() factorises a dense matrix
KAPPA = 1.0         # thermal diffusivity of the non-dimensional equations
TIGHT = dict(rtol_Pat=0.8e-6, rtol_U_final=5e-7)  # a solve to a relative residual of 1e-6


def _shell(kind, level, nlayer, nmg, **kw):
    return dict(kind=kind, mesh="shell", level=level, nlayer=nlayer, nmg=nmg, contrast=1e4, **kw)


def listed():
    return [
        # the smallest Stokes solve of the tests (17k velocity unknowns), all in double: latency and launches decide
        dict(_shell("solve", 1, 2, 2, precision="fp64"), name="solve_small_fp64", contrast=1e3),
        # the reference's own call on a million unknowns: double precision, host arrays in and out, from nothing
        dict(_shell("solve", 2, 4, 3, precision="fp64"), name="solve_1m_fp64"),
        # an unstructured mesh with a refined region and a large coarse grid, mixed precision, from nothing
        dict(kind="solve", mesh="file", level=0, nlayer=0, nmg=2, contrast=1e3, precision="mixed", name="solve_file_mixed"),
        # one step of the time loop with everything in device memory: the learned start, mixed precision
        dict(_shell("step", 2, 4, 3, precision="mixed", start="learned"), name="step_1m_mixed_learned"),
        # the same step from the extrapolation in time, in double precision
        dict(_shell("step", 2, 4, 3, precision="fp64", start="extrapolated"), name="step_1m_fp64"),
        # one velocity solve alone, a million unknowns, double
        dict(_shell("velocity", 2, 4, 3, precision="fp64"), name="velocity_1m_fp64"),
        # one velocity solve alone, eight million unknowns, four levels, mixed
        dict(_shell("velocity", 2, 4, 4, precision="mixed"), name="velocity_8m_mixed"),
        # the operators of a step: element integration, Galerkin products, coarse factorisation, one coarse solve
        dict(_shell("operators", 2, 4, 3), name="operators_1m"),
        # the same on the mesh file, whose coarse factorisation is the largest part
        dict(kind="operators", mesh="file", level=0, nlayer=0, nmg=2, contrast=1e3, name="operators_file"),
        # the temperature's part of a step: diffusion, advection, diffusion on the vertices
        dict(_shell("thermal", 2, 4, 3), name="thermal_1m"),
        # four training steps of the warm-start network: forward, backward, Adam
        dict(_shell("train", 2, 4, 3, steps=4), name="train_1m"),
        # the warm start of one step: extrapolation in time and the network's forward pass
        dict(_shell("start", 2, 4, 3), name="start_1m"),
    ]


def _tets(level, nlayer, nmg):
    return 20 * 4 ** level * 3 * nlayer * 8 ** (nmg - 1)


def draw(rng):
    kind = rng.choice(["solve", "solve", "step", "velocity", "velocity", "operators", "thermal", "train", "start"])
    most = dict(solve=400e3, step=400e3, velocity=1.2e6, operators=400e3, thermal=1.2e6, train=400e3, start=1.2e6)[kind]
    shapes = [(lv, nl, nm) for lv in (1, 2) for nl in range(1, 7) for nm in (2, 3, 4) if _tets(lv, nl, nm) <= most]
    # spread over the logarithm of the size: the shape nearest to a drawn size
    size = 10 ** rng.uniform(np.log10(1900.0), np.log10(most))
    level, nlayer, nmg = min(shapes, key=lambda s: (abs(np.log(_tets(*s) / size)) + 0.1 * rng.random()))
    c = _shell(kind, level, nlayer, nmg)
    c["contrast"] = round(10 ** rng.uniform(2.0, 5.0), 1)
    if kind in ("solve", "step", "velocity"):
        c["precision"] = rng.choice(["fp64", "mixed"])
    if kind == "step":
        c["start"] = rng.choice(["learned", "extrapolated"])
    if kind == "train":
        c["steps"] = rng.randint(1, 6)
    return c


# ---- inputs ------------------------------------------------------------------------------------------------------------------

@functools.lru_cache(maxsize=4)
def _mesh(kind, level, nlayer, nmg):
    if kind == "file":
        return meshmod.build_from_file(MESH_FILE, nmg, device=0)
    return meshmod.build_shell(level, nlayer, nmg, device=0)


def _mesh_of(case):
    return _mesh(case["mesh"], case["level"], case["nlayer"], case["nmg"])


def _harmonics(m, rng, n=24, lmax=8):
    """A random combination of spherical harmonics of degree 1..lmax (zonal ones about random axes), largest value 1, on the nodes."""
    X = torch.from_numpy(m.GCOORD).cuda()
    X = X / X.norm(dim=1, keepdim=True)
    f = torch.zeros(len(X), dtype=torch.float64, device="cuda")
    for _ in range(n):
        c = rng.standard_normal(3)
        t = X @ torch.from_numpy(c / np.linalg.norm(c)).cuda()
        l = int(rng.integers(1, lmax + 1))
        a, b = torch.ones_like(t), t
        for k in range(1, l):
            a, b = b, ((2 * k + 1) * t * b - k * a) / (k + 1)
        f += float(rng.standard_normal()) / (l + 1) * b
    return (f / f.abs().max()).cpu().numpy()


def _temperature(m, rng, amp=0.05):
    """A conductive profile with a perturbation that vanishes on both boundaries."""
    s = (m.r_surf - m.GCOORD_SPH[:, 2]) / (m.r_surf - m.r_cmb)
    return s + amp * _harmonics(m, rng) * np.sin(np.pi * s)


def _material(T, contrast):
    return np.exp(-np.log(contrast) * T), 1.5 - T


def _frames(X):
    """Per node the unit vectors (theta, phi, r) as columns."""
    x, y, z = X.T
    s = np.hypot(x, y)
    r = np.sqrt(x * x + y * y + z * z)
    ct, st = z / r, s / r
    pole = s == 0
    cp, sp = np.where(pole, 1.0, x / np.where(pole, 1, s)), np.where(pole, 0.0, y / np.where(pole, 1, s))
    zero = np.zeros_like(ct)
    return np.stack([np.stack([cp * ct, sp * ct, -st], 1), np.stack([-sp, cp, zero], 1), np.stack([cp * st, sp * st, ct], 1)], 2)


def _plates(m, rng, nplate=6):
    """Velocity conditions: free slip at the inner boundary, rotating plates on the outer one (0-based dofs, values)."""
    centre = rng.standard_normal((nplate, 3))
    pole = rng.standard_normal((nplate, 3))
    pole /= np.linalg.norm(pole, axis=1)[:, None]
    inner, outer = np.nonzero(m.PointID == 301)[0], np.nonzero(m.PointID == 306)[0]
    X = m.GCOORD[outer]
    v = np.einsum("nji,nj->ni", _frames(X), np.cross(pole[np.argmax(X @ centre.T, axis=1)], X))
    v[:, 2] = 0.0
    dofs = np.concatenate([3 * inner + 2, (3 * outer[:, None] + np.arange(3)).ravel()])
    vals = np.concatenate([np.zeros(len(inner)), v.ravel()])
    o = np.argsort(dofs)
    return dofs[o], vals[o]


class _DeviceArray:
    """A device array of the library as torch sees it; it keeps its owner."""

    def __init__(self, owner, address, n):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=(n,), typestr="<f8", data=(address, False), version=2)


def _view(owner, address, n):
    return torch.as_tensor(_DeviceArray(owner, address, n), device="cuda")


def _inputs(case, seed):
    m = _mesh_of(case)
    rng = np.random.default_rng(seed)
    T = _temperature(m, rng)
    V, R = _material(T, case["contrast"])
    ifix, vfix = _plates(m, rng)
    return m, rng, T, V, R, ifix, vfix


def _thermal_inputs(case, seed):
    """Vertex temperatures, a flow of rotating shells and cells through the whole depth, a step of half an element."""
    m, rng, T, _, _, _, _ = _inputs(case, seed)
    nV = m.nVnod
    s = (m.GCOORD_SPH[:, 2] - m.r_cmb) / (m.r_surf - m.r_cmb)
    w = rng.standard_normal(3)
    U = np.einsum("nji,nj->ni", _frames(m.GCOORD), np.cross(w / np.linalg.norm(w), m.GCOORD)) * (0.3 + s)[:, None]
    U[:, 2] += 0.7 * _harmonics(m, rng) * np.sin(np.pi * s)
    E, X = m.levels[0].EL2NOD[:, :4], m.GCOORD
    h = min(np.linalg.norm(X[E[:, a]] - X[E[:, b]], axis=1).min() for a in range(4) for b in range(a))
    dt = 0.5 * h / np.linalg.norm(U, axis=1).max()
    ifix = np.nonzero(np.isin(m.PointID[:nV], (301, 306)))[0]
    return m, T[:nV].copy(), U.ravel(), dt, ifix, np.where(m.PointID[ifix] == 301, 1.0, 0.0)


def _states(case, seed, n):
    """n consecutive synthetic states (T at the vertices, viscosity, U, P) of a slow change, and their times."""
    m = _mesh_of(case)
    rng = np.random.default_rng(seed)
    s = (m.GCOORD_SPH[:, 2] - m.r_cmb) / (m.r_surf - m.r_cmb)
    bump = np.sin(np.pi * s)
    fields = [_harmonics(m, rng) for _ in range(4)]
    out = []
    for k in range(n):
        a = 0.02 * k + 0.004 * k * k
        T = 1 - s + 0.05 * bump * (fields[0] * (1 - a) + fields[1] * a)
        U = 300.0 * bump[:, None] * np.stack([fields[1] * (1 + a), fields[2] * (1 - a), fields[0] + a * fields[3]], 1)
        P = 1e4 * (fields[0] + a * fields[2]) * (1 + s)
        V, _ = _material(T, case["contrast"])
        out.append((T[:m.nVnod].copy(), V, U.ravel().copy(), P[:m.nVnod].copy()))
    return m, out, [1e-3 * (k + 0.1 * np.sin(k)) for k in range(n)]


def _context(m, ifix, vfix):
    ctx = api.StokesContext(m)
    ctx.set_bc(ifix, vfix)
    return ctx


def _vertex_edges(E):
    return np.concatenate([E[:, [a, b]] for a in range(4) for b in range(4) if a != b])


def _training(case, seed):
    """Per step the arguments of WarmStartNet.add_sample, and the network's parameters and normalisation."""
    m, st, _ = _states(case, seed, case["steps"] + 1)
    samples = [(b[0], a[0], b[1], a[2], a[3], b[2], b[3]) for a, b in zip(st, st[1:])]
    XY = [_features(m, *s) for s in samples]
    X, Y = (np.concatenate([v[k] for v in XY]) for k in (0, 1))
    norm = np.concatenate([X.mean(0), X.std(0) + 1e-6, np.sqrt((Y ** 2).mean(0))]).astype(np.float32)
    return m, samples, XY, learned.init_params(seed % 2 ** 31), norm


def _features(m, T, T_prev, V, U_prev, P_prev, U_next=None, P_next=None):
    """The network's inputs and targets on the vertices (64 bits)."""
    n = m.nVnod
    u = U_prev.reshape(-1, 3)[:n]
    dT = T - T_prev
    su, sp, st = np.sqrt((u ** 2).sum() / n), np.sqrt((P_prev ** 2).mean()), np.sqrt((dT ** 2).mean())
    r = np.linalg.norm(m.GCOORD[:n], axis=1)
    X = np.column_stack([T, np.log(V[:n]), u / su, P_prev / sp, (r - m.r_cmb) / (m.r_surf - m.r_cmb), dT / st])
    if U_next is None:
        return X, (su, sp, st)
    return X, np.column_stack([(U_next.reshape(-1, 3)[:n] - u) / (su * st), (P_next - P_prev) / (sp * st)])


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("solve", "operators", "velocity"):
        m, rng, T, V, R, ifix, vfix = _inputs(case, seed)
        s = dict(kind=kind, ctx=_context(m, ifix, vfix), V=V, R=R, case=case)
        if kind == "operators":
            s["rhs"] = rng.standard_normal(3 * m.levels[-1].nnod)
        if kind == "velocity":  # the first velocity solve of a step: its right-hand side without the pressure
            ctx = s["ctx"]
            ctx.assemble(V, R, PHYS)
            ctx.restrict_stiffmat()
            ctx.cholesky_factorization()
            s["b"] = ctx.get_vector(0) - ctx.get_vector(1)
        return s
    if kind == "step":
        m, rng, T, V, R, ifix, vfix = _inputs(case, seed)
        ctx = _context(m, ifix, vfix)
        net = learned.WarmStartNet(m)
        net.load(NETWORK)
        E, X = m.levels[0].EL2NOD[:, :4], m.GCOORD
        h = min(np.linalg.norm(X[E[:, a]] - X[E[:, b]], axis=1).min() for a in range(4) for b in range(a))
        Tv, t, par = T[:m.nVnod].copy(), 0.0, net.edge_parent
        opts = dict(precision=case["precision"], rtol_U_final=5e-7, rtol_U_first=4e-7)
        for k in range(4):
            Tn = np.concatenate([Tv, 0.5 * (Tv[par[:, 0]] + Tv[par[:, 1]])])
            V, R = _material(Tn, case["contrast"])
            if k == 3:
                break
            if k == 0:
                U, P, info = ctx.flow3d(V, R, PHYS, precision="mixed", **TIGHT)
                opts["tol_Pat_abs"] = 0.8e-6 * info["norm_rP0"]
            else:
                _, U0, P0 = net.extrapolate(t, k - 1)
                U, P, info = ctx.flow3d(V, R, PHYS, U0=U0, P0=P0, **dict(opts, precision="mixed"))
            net.push_state(t, Tv, U, P)
            dt = 0.5 * h / np.linalg.norm(U.reshape(-1, 3)[:m.nVnod], axis=1).max()
            Tv = ctx.sl_advect(Tv, U, dt)
            t += dt
        ctx.set_fields(V, R)
        net.set_inputs(Tv, V)
        return dict(kind=kind, ctx=ctx, net=net, t=t, opts=opts, case=case)
    if kind == "thermal":
        m, T, U, dt, ifix, vfix = _thermal_inputs(case, seed)
        ctx = api.StokesContext(m)
        ctx.diffusion_mesh()
        return dict(kind=kind, ctx=ctx, T=T, U=U, dt=dt, ifix=ifix, vfix=vfix, case=case)
    if kind == "train":
        m, samples, _, params, norm = _training(case, seed)
        net = learned.WarmStartNet(m)
        net.set_params(params, norm)
        net.reserve(len(samples))
        for i, a in enumerate(samples):
            net.add_sample(i, *a)
        return dict(kind=kind, net=net, ids=np.arange(len(samples)), case=case)
    if kind == "start":
        m, st, ts = _states(case, seed, 4)
        net = learned.WarmStartNet(m)
        net.load(NETWORK)
        for (T, _, U, P), t in zip(st[:3], ts):
            net.push_state(t, T, U, P)
        net.set_inputs(st[3][0], st[3][1])
        return dict(kind=kind, net=net, t=ts[3], case=case)
    raise ValueError(kind)


# ---- one pass ----------------------------------------------------------------------------------------------------------------

def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "solve":
        U, P, _ = s["ctx"].flow3d(s["V"], s["R"], PHYS, precision=case["precision"], **TIGHT)
        return dict(U=U, P=P)
    if kind == "step":
        ctx, net = s["ctx"], s["net"]
        if case["start"] == "learned":
            net.solve(ctx, s["t"], 2, PHYS, keep_on_device=True, **s["opts"])
        else:
            net.extrapolate(s["t"], 2, device=True)
            ctx.flow3d(None, None, PHYS, start_device=net.start_device(), keep_on_device=True, **s["opts"])
        u, p = ctx.solution_device()
        return dict(U=_view(s, u, 3 * ctx.mesh.nnod), P=_view(s, p, ctx.mesh.nVnod))
    if kind == "velocity":
        x, _, _ = s["ctx"].mgpcg(s["b"], tol=1e-8, is_abs_tol=False, itmax=60, precision=case["precision"])
        return x
    if kind == "operators":
        ctx = s["ctx"]
        ctx.assemble(s["V"], s["R"], PHYS)
        ctx.restrict_stiffmat()
        ctx.cholesky_factorization()
        return ctx.cholesky_solve(s["rhs"])
    if kind == "thermal":
        ctx, dt = s["ctx"], s["dt"]
        T, _ = ctx.diffusion3d(s["T"], KAPPA, dt / 2, s["ifix"], s["vfix"])
        T = ctx.sl_advect(T, s["U"], dt, 1.0, 0.0)
        T, _ = ctx.diffusion3d(T, KAPPA, dt / 2, s["ifix"], s["vfix"])
        return T
    if kind == "train":
        loss = s["net"].train(s["ids"], 1e-3)
        params, _ = s["net"].get_params()
        return dict(loss=loss, params=params)
    net = s["net"]
    net.warm_start_hist(s["t"], 2, None, None, device=True)
    u, p = net.start_device()
    return dict(U=_view(s, u, 3 * net.mesh.nnod), P=_view(s, p, net.n))


# ---- the work of one pass ----------------------------------------------------------------------------------------------------

# CG iterations of a solve of each kind on a million unknowns, to price it (a pass takes more or fewer with its viscosity)
ITERATIONS = dict(solve=200, step=70, velocity=17)


def work(case):
    nel = 210880 if case["mesh"] == "file" else _tets(case["level"], case["nlayer"], case["nmg"])
    base = 26360 if case["mesh"] == "file" else nel // 8 ** (case["nmg"] - 1)
    nV = nel / 6.0 + 300          # vertices and P2 nodes of a shell of nel tetrahedra
    nn = 1.36 * nel + 2000
    blocks = 28.0 * nn            # 3x3 blocks of the velocity operator
    kind = case["kind"]
    if kind == "train":
        dense = nV * 2 * (8 * 64 + 3 * 128 * 64 + 64 * 4)
        return dict(flops=3.0 * dense * case["steps"], bytes=case["steps"] * nV * (12 * 4 + 10 * 64 * 2 * 2.0))
    if kind == "start":
        return dict(flops=nV * 2 * (8 * 64 + 3 * 128 * 64 + 64 * 4), bytes=8.0 * (4 * (3 * nn + 2 * nV)) + nV * 7 * 64 * 2 * 2.0)
    if kind == "thermal":  # two systems of 14 entries a row and about 20 iterations each, the advection
        return dict(flops=nel * 2 * 4 * 400.0 + 40 * nV * 2 * 14, bytes=2 * (nel * 16 + 20 * nV * (14 * 12 + 8 * 8)) + nel * 16 + nV * 100.0)
    # operators: 14 points of a 30x30 matrix, K written once, the products down the levels, the coarse factor
    nc3 = 3 * (1.36 * base + 1000)
    flops = nel * (14 * 55 * 9 * 4.0 + 8 / 7 * 55 * 9 * 10 * 2) + 40.0 * nc3 ** 2
    bytes_ = nel * 40.0 + blocks * 72 * 8 / 7 + nc3 * 8 * 900
    if kind != "operators":
        it = ITERATIONS[kind]
        vb = 76.0 if case["precision"] == "fp64" else 24.0
        each = blocks * (76 + 7 * 8 / 7 * vb) + nn * 3 * 8 * 20
        op = (0.0, 0.0) if kind == "velocity" else (flops, bytes_)
        return dict(flops=op[0] + it * blocks * 9 * 18.0, bytes=op[1] + it * each)
    return dict(flops=flops, bytes=bytes_)


def tolerance(case):
    return {
        # stopped at a residual of 1e-6: FP64 and mixed V-cycles end up to 5e-5 apart at the high viscosity contrasts
        "solve": dict(rel=2e-4, max=2e-2), "step": dict(rel=2e-4, max=2e-2),
        # stopped at 1e-8: 6e-10 from the dense solution, and one iteration more or less is about ten times that
        "velocity": dict(rel=4e-8, max=2e-6),
        # 64 bits throughout, sums in any order: 2e-15 from the dense solution, times the contrast's conditioning
        "operators": dict(rel=1e-12, max=1e-10),
        # conjugate gradients stopped at 1e-8 twice: 3e-10 from the solution
        "thermal": dict(rel=2e-9, max=1e-7),
        # 16-bit activations: parameters 4e-4 from 64 bits after four steps (Adam turns a small gradient's sign into a step)
        "train": dict(rel=1.6e-3, max=0.1),
        # the network's correction in 32 bits on 16-bit activations, a small part of the state: 5e-7
        "start": dict(rel=2e-6, max=1e-4),
    }[case["kind"]]


# ---- the same in 64 bits, in plain torch -------------------------------------------------------------------------------------

def _cart2sph(X):
    x, y, z = X.unbind(-1)
    ph = torch.atan2(y, x)
    return torch.stack([torch.atan2(torch.hypot(x, y), z), torch.where(ph < 0, ph + 2 * np.pi, ph), torch.sqrt(x * x + y * y + z * z)], -1)


def _bary_derivatives(f, L):
    """f and its derivatives with respect to the first three barycentric coordinates (the fourth is one minus their sum), per point."""
    out, d = [], []
    for l in L:
        v = f(l)
        g = torch.autograd.functional.jacobian(f, l)
        out.append(v)
        d.append(g[:, :3] - g[:, 3:])
    return torch.stack(out), torch.stack(d)


EDGES10 = ((0, 1), (1, 2), (2, 3), (3, 0), (0, 2), (3, 1))
EDGES20 = ((0, 1), (1, 2), (2, 3), (3, 0), (0, 2), (3, 1))  # two nodes each, the one nearer the first vertex first


def _n10(l):
    return torch.stack([l[i] * (2 * l[i] - 1) for i in range(4)] + [4 * l[a] * l[b] for a, b in EDGES10])


def _n20(l):
    e = [4.5 * l[a] * l[b] * (3 * l[k] - 1) for a, b in EDGES20 for k in (a, b)]
    return torch.stack([0.5 * l[i] * (3 * l[i] - 1) * (3 * l[i] - 2) for i in range(4)] + e +
                       [27 * l[1] * l[2] * l[3], 27 * l[0] * l[2] * l[3], 27 * l[0] * l[1] * l[3], 27 * l[0] * l[1] * l[2]])


def _rule14():
    """The 14-point rule of degree 5: barycentric points and weights (their sum is 1/6)."""
    g = 1 / (46 * np.sqrt(46))
    k = (104 + 8 * np.sqrt(46) * np.cos(np.arccos(g) + 2 / 3 * np.arcsin(g))) / 3
    s = np.sqrt(49 - k)
    b, d = (7 + s) / k, (7 - s) / k
    a, c = 1 - 3 * b, 1 - 3 * d
    p, q = (98 - k - 14 * s) / (1680 * s * (b - a) ** 3), (98 - k + 14 * s) / (1680 * s * (c - d) ** 3)
    r = (1 - 4 * (p + q)) / 6
    e = (1 + (2 / (105 * r)) ** 0.25) / 4
    f = (1 - 2 * e) / 2
    L = [[a if i == j else b for j in range(4)] for i in range(4)] + [[c if i == j else d for j in range(4)] for i in range(4)]
    L += [[e if j in ij else f for j in range(4)] for ij in ((0, 1), (0, 2), (0, 3), (1, 2), (1, 3), (2, 3))]
    return L, [p / 6] * 4 + [q / 6] * 4 + [r / 6] * 6


# the frames in which elements are mapped: original, turned about z by pi, turned about x by a quarter
TURN = dict(out_cone_no_cross_2pi=[[1, 0, 0], [0, 1, 0], [0, 0, 1]], out_cone_cross_2pi=[[-1, 0, 0], [0, -1, 0], [0, 0, 1]],
            in_cone_no_iso=[[1, 0, 0], [0, 0, -1], [0, 1, 0]], in_cone_iso=[[1, 0, 0], [0, 0, -1], [0, 1, 0]])


def _points(m, els, name, iso_at, L, dev, straight=False):
    """At every point of every element of one class: Cartesian derivatives map (inverse Jacobian, columns by barycentric coordinate),
    determinant and the outward unit vector."""
    Q = torch.tensor(TURN[name], dtype=torch.float64, device=dev)
    if name == "in_cone_iso" and not straight:
        S = _cart2sph(torch.from_numpy(m.X20_iso[iso_at]).to(dev) @ Q.T)
        N, dN = _bary_derivatives(_n20, L)
    else:
        E = m.levels[0].EL2NOD[els, :4]
        if name in ("out_cone_no_cross_2pi", "out_cone_cross_2pi"):
            S = torch.from_numpy(m.GCOORD_SPH[E]).to(dev).clone()
            if name == "out_cone_cross_2pi":
                ph = S[..., 1] + np.pi
                S[..., 1] = torch.where(ph > 2 * np.pi, ph - 2 * np.pi, ph)
        else:
            S = _cart2sph(torch.from_numpy(m.GCOORD[E]).to(dev) @ Q.T)
        N, dN = _bary_derivatives(lambda l: l, L)
    N, dN = N.to(dev), dN.to(dev)
    for p in range(len(L)):
        th, ph, r = torch.einsum("k,ekc->ec", N[p], S).unbind(-1)
        st, ct, sp, cp = th.sin(), th.cos(), ph.sin(), ph.cos()
        up = torch.stack([st * cp, st * sp, ct], -1)
        dX = torch.stack([torch.stack([r * ct * cp, r * ct * sp, -r * st], -1), torch.stack([-r * st * sp, r * st * cp, 0 * r], -1), up], -1)
        J = dX @ torch.einsum("ekc,kj->ecj", S, dN[p])
        yield p, torch.linalg.inv(J) @ Q, torch.linalg.det(J).abs(), up @ Q


def _elements(m, els, name, iso_at, V, R, dev):
    """Element matrices of some elements of one class: K (n,30,30), G (n,30,4), F (n,30)."""
    L, w = _rule14()
    L = [torch.tensor(l, dtype=torch.float64) for l in L]
    N10, d10 = (t.to(dev) for t in _bary_derivatives(_n10, L))
    E = torch.from_numpy(m.levels[0].EL2NOD[els, :4]).to(dev)
    eye = torch.eye(3, dtype=torch.float64, device=dev)
    K, G, F = 0, 0, 0
    for p, iJ, det, up in _points(m, els, name, iso_at, L, dev):
        l = L[p].to(dev)
        D = d10[p] @ iJ
        c = det * w[p]
        k = c * (V[E] @ l)
        DD = torch.einsum("eai,ebj->eaibj", D, D)
        same = torch.einsum("eaibi->eab", DD)
        K = K + k[:, None, None, None, None] * (DD.transpose(2, 4) - 2 / 3 * DD + same[:, :, None, :, None] * eye[None, None, :, None, :])
        G = G + (c[:, None, None, None] * D[..., None] * l).reshape(-1, 30, 4)
        F = F + (PHYS["g"] * PHYS["Bscale"] * c * (R[E] @ l - PHYS["Dens0"]))[:, None] * torch.einsum("a,ei->eai", N10[p], up).reshape(-1, 30)
    return K.reshape(-1, 30, 30), G, F


def _assembled(m, V, R, dev, chunk=20000):
    """Every element's matrices in the nodes' (theta, phi, r) frames, in pieces: (elements, K, G, F)."""
    V, R = torch.from_numpy(V).to(dev), torch.from_numpy(R).to(dev)
    fr = torch.from_numpy(_frames(m.GCOORD)).to(dev)
    for name in TURN:
        every = m.classes[name]
        for i in range(0, len(every), chunk):
            els = every[i:i + chunk]
            K, G, F = _elements(m, els, name, slice(i, i + chunk), V, R, dev)
            E = torch.from_numpy(m.levels[0].EL2NOD[els]).to(dev)
            f = fr[E]
            K = torch.einsum("eaji,eajbk,ebkl->eaibl", f, K.reshape(-1, 10, 3, 10, 3), f).reshape(-1, 30, 30)
            G = torch.einsum("eaji,eajv->eaiv", f, G.reshape(-1, 10, 3, 4)).reshape(-1, 30, 4)
            F = torch.einsum("eaji,eaj->eai", f, F.reshape(-1, 10, 3)).reshape(-1, 30)
            yield torch.from_numpy(els).to(dev), E, K, G, F


def _dofs(E):
    return (3 * E[:, :, None] + torch.arange(3, device=E.device)).reshape(len(E), -1)


def _dense(m, V, R, dev):
    n, nV = 3 * m.nnod, m.nVnod
    K, G, F = (torch.zeros(s, dtype=torch.float64, device=dev) for s in ((n * n,), (n * nV,), (n,)))
    for _, E, Ke, Ge, Fe in _assembled(m, V, R, dev):
        d = _dofs(E)
        K.index_add_(0, (d[:, :, None] * n + d[:, None, :]).reshape(-1), Ke.reshape(-1))
        G.index_add_(0, (d[:, :, None] * nV + E[:, None, :4]).reshape(-1), Ge.reshape(-1))
        F.index_add_(0, d.reshape(-1), Fe.reshape(-1))
    return K.reshape(n, n), G.reshape(n, nV), F


def _exact_flow(case, seed, dev, velocity_only):
    m, _, _, V, R, ifix, vfix = _inputs(case, seed)
    if 3 * m.nnod > DENSE:
        return None
    K, G, F = _dense(m, V, R, dev)
    U0 = torch.zeros(3 * m.nnod, dtype=torch.float64, device=dev)
    U0[torch.from_numpy(ifix).to(dev)] = torch.from_numpy(vfix).to(dev)
    free = torch.ones_like(U0, dtype=torch.bool)
    free[torch.from_numpy(ifix).to(dev)] = False
    C = torch.linalg.cholesky(K[free][:, free])
    f, Gf = (F - K @ U0)[free], G[free]
    x = torch.cholesky_solve(f[:, None], C)[:, 0]
    if velocity_only:
        U = torch.zeros_like(U0)
        U[free] = x
        return U.cpu()
    B = torch.cholesky_solve(Gf, C)
    S = Gf.T @ B + 1.0 / m.nVnod  # constant pressures: the solver's have mean zero
    r = -(G.T @ U0) - Gf.T @ x
    P = torch.linalg.solve(S, r - r.mean())
    P -= P.mean()
    U0[free] += x + B @ P
    return dict(U=U0.cpu(), P=P.cpu())


def _children(m, l, dev):
    """Per element of level l the weights (10, 10) of its parent's nodes at its nodes."""
    ptr, col, w = m.transfer(l)
    n, ptr = m.levels[l].nnod, np.asarray(ptr)
    at = ptr[:-1, None] + np.arange(10)
    has = at < ptr[1:, None]
    at = np.minimum(at, len(col) - 1)
    c = torch.from_numpy(np.where(has, np.asarray(col)[at], -1)).to(dev)
    ww = torch.from_numpy(np.where(has, np.asarray(w)[at], 0.0)).to(dev)
    E = torch.from_numpy(m.levels[l].EL2NOD).to(dev)
    Ec = torch.from_numpy(m.levels[l + 1].EL2NOD).to(dev)
    for i in range(0, len(E), 16000):
        e = E[i:i + 16000]
        parent = torch.arange(i, i + len(e), device=dev) // 8
        same = (c[e][:, :, :, None] == Ec[parent][:, None, None, :]).double()
        yield slice(i, i + len(e)), parent, torch.einsum("eak,eakb->eab", ww[e], same)


def _exact_operators(case, seed, dev):
    m, rng, _, V, R, ifix, vfix = _inputs(case, seed)
    rhs = torch.from_numpy(rng.standard_normal(3 * m.levels[-1].nnod)).to(dev)
    if 3 * m.levels[-1].nnod > DENSE or m.nel > 500000:
        return None
    free = torch.ones(3 * m.nnod, dtype=torch.float64, device=dev)
    free[torch.from_numpy(ifix).to(dev)] = 0.0
    Ke = torch.zeros((m.nel, 30, 30), dtype=torch.float64, device=dev)
    for els, E, K, _, _ in _assembled(m, V, R, dev):
        d = free[_dofs(E)]
        Ke[els] = K * d[:, :, None] * d[:, None, :]
    for l in range(m.nmg - 1):
        Kc = torch.zeros((len(m.levels[l + 1].EL2NOD), 30, 30), dtype=torch.float64, device=dev)
        for i, parent, Q in _children(m, l, dev):
            Kc.index_add_(0, parent, torch.einsum("eap,eaibj,ebq->epiqj", Q, Ke[i].reshape(-1, 10, 3, 10, 3), Q).reshape(-1, 30, 30))
        d = free[_dofs(torch.from_numpy(m.levels[l + 1].EL2NOD).to(dev))]
        Ke = Kc * d[:, :, None] * d[:, None, :]
    n = 3 * m.levels[-1].nnod
    A = torch.diag(1 - free[:n]).reshape(-1)
    d = _dofs(torch.from_numpy(m.levels[-1].EL2NOD).to(dev))
    A.index_add_(0, (d[:, :, None] * n + d[:, None, :]).reshape(-1), Ke.reshape(-1))
    return (torch.linalg.solve(A.reshape(n, n), rhs * free[:n])).cpu()


def _diffuse(A, M, T, ifix, vfix):
    """One implicit step (M + A) T' = M T with fixed values, by conjugate gradients to the end."""
    T = T.clone()
    b = M * T
    T[ifix] = vfix
    free = torch.ones_like(T)
    free[ifix] = 0.0
    op = lambda v: M * v + A(v)  # noqa: E731
    r = (b - op(T)) * free
    q = z = r / M
    rz, first = r @ z, (r @ z).clone()
    for _ in range(400):
        if rz <= 1e-32 * first:
            break
        Aq = op(q) * free
        a = rz / (q @ Aq)
        T, r = T + a * q, r - a * Aq
        z = r / M
        rz, old = r @ z, rz
        q = z + (rz / old) * q
    return T


def _exact_thermal(case, seed, dev):
    m, T, U, dt, ifix, vfix = _thermal_inputs(case, seed)
    n, E, X = m.nVnod, m.levels[0].EL2NOD[:, :4], m.GCOORD[:m.nVnod]
    if m.nel > 500000:
        return None
    # linear elements, mapped in the same frames as their classes by vertices, four points
    tc = np.deg2rad(m.theta_cone)
    th, ph = m.GCOORD_SPH[E, 0], m.GCOORD_SPH[E, 1]
    cone = ((th <= tc) | (th >= np.pi - tc)).sum(1) > 0
    cross = (ph.max(1) - ph.min(1)) > np.pi
    groups = dict(out_cone_no_cross_2pi=~cone & ~cross, out_cone_cross_2pi=~cone & cross, in_cone_no_iso=cone)
    a, b = (5 + 3 * np.sqrt(5)) / 20, (5 - np.sqrt(5)) / 20
    L = [torch.tensor([a if i == j else b for j in range(4)], dtype=torch.float64) for i in range(4)]
    d4 = torch.tensor([[1., 0, 0], [0, 1, 0], [0, 0, 1], [-1, -1, -1]], dtype=torch.float64, device=dev)
    Ce, Me = torch.zeros((len(E), 4, 4), dtype=torch.float64, device=dev), torch.zeros((len(E), 4), dtype=torch.float64, device=dev)
    for name, mask in groups.items():
        els = np.nonzero(mask)[0]
        if len(els):
            at = torch.from_numpy(els).to(dev)
            for p, iJ, det, _ in _points(m, els, name, None, L, dev, straight=True):
                D = d4 @ iJ
                Ce[at] += (det / 24)[:, None, None] * (D @ D.transpose(1, 2))
                Me[at] += (det / 24)[:, None] * L[p].to(dev)
    Et = torch.from_numpy(E).to(dev)
    M = torch.zeros(n, dtype=torch.float64, device=dev).index_add_(0, Et.reshape(-1), Me.reshape(-1))
    A = lambda v: 0.5 * dt * KAPPA * torch.zeros_like(v).index_add_(0, Et.reshape(-1), torch.einsum("eab,eb->ea", Ce, v[Et]).reshape(-1))  # noqa: E731
    fix, val = torch.from_numpy(ifix).to(dev), torch.from_numpy(vfix).to(dev)
    T = _diffuse(A, M, torch.from_numpy(T).to(dev), fix, val)
    T = _advect(m, Et, torch.from_numpy(X).to(dev), T, torch.from_numpy(U.reshape(-1, 3)[:n]).to(dev), dt, fix, val)
    return _diffuse(A, M, T, fix, val).cpu()


def _advect(m, E, X, T, U, dt, fix, val):
    """Midpoint back-tracking along great circles and linear interpolation in the straight tetrahedra around each vertex."""
    n, dev = len(X), X.device
    u = torch.einsum("nij,nj->ni", torch.from_numpy(_frames(m.GCOORD[:n])).to(dev), U)
    order = torch.argsort(E.reshape(-1), stable=True)
    count = torch.bincount(E.reshape(-1), minlength=n)
    first = torch.cumsum(count, 0) - count
    S = int(count.max())
    at = first[:, None] + torch.arange(S, device=dev)
    star = torch.where(torch.arange(S, device=dev) < count[:, None], order[at.clamp(max=len(order) - 1)] // 4, -1)
    x4 = X[E[:, 3]]
    inv = torch.linalg.inv(torch.stack([X[E[:, k]] - x4 for k in range(3)], -1))
    rad = X.norm(dim=1)
    xh = X / rad[:, None]

    def best_of(p, cand):
        l = torch.einsum("vcij,vcj->vci", inv[cand.clamp(min=0)], p[:, None] - x4[cand.clamp(min=0)])
        l = torch.cat([l, 1 - l.sum(-1, keepdim=True)], -1)
        low = torch.where(cand >= 0, l.min(-1).values, -torch.inf)
        k = low.argmax(1, keepdim=True)
        return low.gather(1, k)[:, 0], cand.gather(1, k)[:, 0], l.gather(1, k[:, :, None].expand(-1, -1, 4))[:, 0]

    def interpolate(p, f):
        low, tet, l = best_of(p, star)
        far = torch.nonzero(low < -1e-12)[:, 0]
        if len(far):
            cand = torch.cat([tet[far, None], star[E[tet[far]]].reshape(len(far), -1)], 1)
            low[far], tet[far], l[far] = best_of(p[far], cand)
        c = l.clamp(min=0)
        l = torch.where((low < 0)[:, None], c / c.sum(1, keepdim=True), l)
        return torch.einsum("vi,vic->vc", l, f[E[tet]])

    def back(w, tau, r_ang, up):
        t = w - (w * xh).sum(1, keepdim=True) * xh
        s = t.norm(dim=1, keepdim=True)
        al = tau * s / r_ang[:, None]
        y = torch.where(s > 0, al.cos() * xh - al.sin() * t / s.clamp(min=1e-300), xh)
        return (rad - tau * (w * up).sum(1)).clamp(rad.min(), rad.max())[:, None] * y

    xm = back(u, 0.5 * dt, rad, xh)
    rm = xm.norm(dim=1)
    out = interpolate(back(interpolate(xm, u), dt, rm, xm / rm[:, None]), T[:, None])[:, 0]
    out[fix] = val
    return out


def _network(p, norm, X, E, n):
    """The network's output for features X (n, 8), differentiable in p."""
    at = 0

    def take(*shape):
        nonlocal at
        k = int(np.prod(shape))
        at += k
        return p[at - k:at].reshape(shape)

    h = torch.relu((X - norm[:8]) / norm[8:16] @ take(8, 64) + take(64))
    deg = torch.bincount(E[:, 0], minlength=n).double()[:, None]
    for _ in range(3):
        mean = torch.zeros_like(h).index_add(0, E[:, 0], h[E[:, 1]]) / deg
        h = h + torch.relu(torch.cat([h, mean], 1) @ take(128, 64) + take(64))
    return h @ take(64, 4) + take(4)


def _edges(m, dev):
    pairs = torch.from_numpy(_vertex_edges(m.levels[0].EL2NOD[:, :4])).to(dev)
    key = torch.unique(pairs[:, 0] * m.nVnod + pairs[:, 1])
    return torch.stack([key // m.nVnod, key % m.nVnod], 1)


def _exact_train(case, seed, dev):
    m, _, XY, params, norm = _training(case, seed)
    if m.nVnod > 100000:
        return None
    p, norm = torch.from_numpy(params).double().to(dev).requires_grad_(True), torch.from_numpy(norm).double().to(dev)
    E, losses = _edges(m, dev), []
    adam = torch.optim.Adam([p], lr=1e-3, betas=(0.9, 0.999), eps=1e-8)
    for X, Y in XY:
        X, Y = (torch.from_numpy(v.astype(np.float32)).double().to(dev) for v in (X, Y))
        adam.zero_grad()
        loss = ((_network(p, norm, X, E, m.nVnod) - Y / norm[16:]) ** 2).mean()
        loss.backward()
        adam.step()
        losses.append(float(loss.detach()))
    return dict(loss=np.array(losses), params=p.detach().cpu())


def _exact_start(case, seed, dev):
    m, st, ts = _states(case, seed, 4)
    w = [np.prod([(ts[3] - ts[j]) / (ts[k] - ts[j]) for j in range(3) if j != k]) for k in range(3)]
    T, U, P = (sum(w[k] * st[k][c] for k in range(3)) for c in (0, 2, 3))
    X, (su, sp, s_T) = _features(m, st[3][0], T, st[3][1], U, P)
    z = np.load(NETWORK, allow_pickle=False)
    norm = torch.from_numpy(z["norm"]).double().to(dev)
    with torch.no_grad():
        Y = _network(torch.from_numpy(z["params"]).double().to(dev), norm, torch.from_numpy(X).to(dev), _edges(m, dev), m.nVnod) * norm[16:]
    Y = Y.cpu().numpy()
    n, E = m.nVnod, m.levels[0].EL2NOD
    par = np.zeros((m.nnod, 2), dtype=np.int64)
    par[:n] = np.arange(n)[:, None]
    for k, (a, b) in enumerate(EDGES10):
        par[E[:, 4 + k]] = E[:, [a, b]]
    dU = Y[:, :3] * (su * s_T)
    return dict(U=U + (0.5 * (dU[par[:, 0]] + dU[par[:, 1]])).ravel(), P=P + Y[:, 3] * (sp * s_T))


def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    kind = case["kind"]
    if kind in ("solve", "velocity"):
        return _exact_flow(case, seed, dev, kind == "velocity")
    if kind == "operators":
        return _exact_operators(case, seed, dev)
    if kind == "thermal":
        return _exact_thermal(case, seed, dev)
    if kind == "train":
        return _exact_train(case, seed, dev)
    if kind == "start":
        return _exact_start(case, seed, dev)
    return None  # a step starts from solves of its own: its result in 64 bits would take a whole trajectory
