"""Performance cases of the pressure-Poisson path, each through the public entry points.

listed() holds the cases, draw() more of the same ranges; prepare() makes what a
solver's time step has in hand (vectors of one seed, and the mesh's handle),
run() is one pass, exact() the same outputs in 64 bits in plain torch.

A program sets one mesh up and applies its handle to many vectors, so the
handle of the case in use is kept here and shared by the states of all seeds."""
import json
import math

import numpy as np
import torch

import nekrs_amd

# solver options by name: the ones of the benchmark's solves
SOLVES = {
    # plain Poisson, Jacobi-preconditioned CG, all FP64
    "jacobi": dict(precon="jacobi", solver="pcg", tol=1e-8, max_iter=1000),
    # the pressure defaults: flexible GMRES(15), FP32 p-multigrid N-3-1 with the
    # restricted Schwarz smoother, one AMG-preconditioned CG iteration at the bottom
    "mixed-ras": dict(precon="multigrid", solver="fgmres", gmresRestart=15, tol=1e-8, max_iter=200,
                      smoother="opt4chebyshev+ras", cheby_degree=3, mgPrecision=0, coarse="amg",
                      coarse_tol=0.0, coarse_max_iter=1),
    # additive Schwarz with the box solves in BF16, as the Helmholtz batch has it
    "mixed-asm-bf16": dict(precon="multigrid", solver="fcg", tol=1e-8, max_iter=500,
                           smoother="opt4chebyshev+asm", cheby_degree=3, mgPrecision=0, fdmPrecision=1,
                           coarse="amg", coarse_tol=0.0, coarse_max_iter=2),
    # the FP64 p-multigrid with Chebyshev-Jacobi smoothing
    "fp64-chebyshev": dict(precon="multigrid", solver="fcg", tol=1e-8, max_iter=1000,
                           smoother="chebyshev+jacobi", cheby_degree=2, mgPrecision=1, coarse="amg",
                           coarse_tol=0.0, coarse_max_iter=2),
}


def listed():
    return [
        # the smallest operator calls: a coarse test mesh, where the launches are what counts
        dict(name="operator 4^3 N7", op="operator", N=7, nx=4, ny=4, nz=4, map="kershaw", fields=1, lambda1=0.0),
        # the benchmark's headline: Ax and gather-scatter at 32^3, order 7
        dict(name="operator 32^3 N7", op="operator", N=7, nx=32, ny=32, nz=32, map="kershaw", fields=1, lambda1=0.0),
        # Helmholtz operators of other orders, as in the benchmark's batch (N in 3, 5, 7, 9), odd boxes
        dict(name="helmholtz 19x18x20 N9", op="operator", N=9, nx=19, ny=18, nz=20, map="kershaw", fields=1,
             lambda1=5.0),
        # the velocity operator: three fields at once, on curved elements
        dict(name="velocity 19x17x18 N5", op="operator", N=5, nx=19, ny=17, nz=18, map="sine", fields=3,
             lambda1=10.0),
        # averaging a vector field over shared nodes: gather-scatter of three vectors
        dict(name="average 21x20x22 N7 x3", op="average", N=7, nx=21, ny=20, nz=22, map="none", dtype="f64", nvec=3),
        # the pressure right-hand side of a time step, at the headline's mesh
        dict(name="pressure rhs 32^3 N7", op="rhs", N=7, nx=32, ny=32, nz=32, map="kershaw"),
        # one application of the Schwarz smoother, FP32 box solves, the published Kershaw mesh
        dict(name="smoother ras 20^3 N7", op="smoother", N=7, nx=20, ny=20, nz=20, map="kershaw", lambda1=0.0,
             options="mixed-ras"),
        # the additive form with BF16 box solves, Helmholtz, order 5, as in the batch
        dict(name="smoother asm 17x19x18 N5", op="smoother", N=5, nx=17, ny=19, nz=18, map="kershaw", lambda1=3.8,
             options="mixed-asm-bf16"),
        # one V-cycle, mixed precision (the pressure defaults) and FP64
        dict(name="vcycle mixed 20^3 N7", op="vcycle", N=7, nx=20, ny=20, nz=20, map="kershaw", lambda1=0.0,
             options="mixed-ras"),
        dict(name="vcycle fp64 24^3 N7", op="vcycle", N=7, nx=24, ny=24, nz=24, map="kershaw", lambda1=0.0,
             options="fp64-chebyshev"),
        # whole solves: the plain Poisson case, and the published Kershaw benchmark
        dict(name="solve jacobi 8^3 N7", op="solve", N=7, nx=8, ny=8, nz=8, map="none", lambda1=0.0,
             options="jacobi"),
        dict(name="solve mixed 20^3 N7", op="solve", N=7, nx=20, ny=20, nz=20, map="kershaw", lambda1=0.0,
             options="mixed-ras"),
    ]


def _box(rng, N, lo, hi):
    """Edges of a near-cubic box of lo to hi elements (over the logarithm), at most hi."""
    E = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    a = E ** (1.0 / 3.0)
    n = [max(2, round(a * rng.uniform(0.8, 1.25))) for _ in range(3)]
    while n[0] * n[1] * n[2] > hi:
        n[n.index(max(n))] -= 1
    return dict(N=N, nx=n[0], ny=n[1], nz=n[2])


def draw(rng):
    op = rng.choice(["operator", "operator", "average", "rhs", "smoother", "vcycle", "solve"])
    orders = [3, 4, 5, 6, 7, 7, 8, 9]
    if op == "operator":
        N = rng.choice(orders)
        fields = rng.choice([1, 1, 3])
        c = dict(op=op, **_box(rng, N, 64, 16777216 // (fields * (N + 1) ** 3)), map=rng.choice(["kershaw", "sine"]),
                 fields=fields)
        return dict(c, lambda1=round(rng.uniform(0.1, 10.0), 3) if fields == 3 else
                    rng.choice([0.0, round(rng.uniform(0.1, 10.0), 3)]))
    if op == "average":
        N = rng.choice(orders)
        return dict(op=op, **_box(rng, N, 64, 8388608 // (N + 1) ** 3), map="none", dtype=rng.choice(["f64", "f32"]),
                    nvec=rng.choice([1, 3]))
    if op == "rhs":
        N = rng.choice(orders)
        return dict(op=op, **_box(rng, N, 216, 8388608 // (N + 1) ** 3), map=rng.choice(["kershaw", "sine"]))
    if op == "solve":
        o = rng.choice(["jacobi", "mixed-ras", "mixed-asm-bf16"])
        N = rng.choice([3, 5, 7, 9])
        if o == "jacobi":
            return dict(op=op, **_box(rng, N, 64, 262144 // (N + 1) ** 3), map="none", lambda1=0.0, options=o)
        return dict(op=op, **_box(rng, N, 216, 2097152 // (N + 1) ** 3), map="kershaw",
                    lambda1=0.0 if o == "mixed-ras" else round(rng.uniform(0.1, 10.0), 3), options=o)
    # the multigrid's smoother and V-cycle: the batch's orders
    N = rng.choice([3, 5, 7, 9])
    o = rng.choice(["mixed-ras", "mixed-asm-bf16"] if op == "smoother" else
                   ["mixed-ras", "mixed-asm-bf16", "fp64-chebyshev"])
    return dict(op=op, **_box(rng, N, 216, 4096000 // (N + 1) ** 3), map="kershaw",
                lambda1=round(rng.uniform(0.1, 10.0), 3) if o == "mixed-asm-bf16" else 0.0, options=o)


# ------------------------------------------------------------------ the cases

class _Setup:
    """One mesh and its handle."""

    def __init__(self, c):
        op, N = c["op"], c["N"]
        self.mesh = m = nekrs_amd.BoxMesh(c["nx"], c["ny"], c["nz"], N, c["map"], 0.3 if c["map"] == "kershaw" else 0.0)
        self.gid = torch.from_numpy(m.gid).cuda()
        self.L = m.Nlocal
        if op == "average":
            self.handle = nekrs_amd.Ogs(m.gid)
            self.weight = self.handle.inv_degree().to(torch.float64 if c["dtype"] == "f64" else torch.float32)
        elif op == "rhs":
            # a channel: inflow at x = 0, outflow at x = 1, walls in y, symmetry in z
            kind = np.array([7, 1, 16, 1, 3, 7], dtype=np.int32)
            bc = np.where(np.asarray(m.EToB).reshape(-1, 6) != 0, kind[None, :], 0).astype(np.int32).ravel()
            self.bc = bc
            self.handle = nekrs_amd.PressureRhs(m, bc)
        else:
            kw = dict(SOLVES[c["options"]]) if "options" in c else dict(precon="jacobi")
            if kw["precon"] == "multigrid" and N in (7, 9):
                kw["levels"] = [N, 3, 1]
            l1 = c["lambda1"]
            self.handle = nekrs_amd.Elliptic(m, lambda0=1.0, lambda1=l1, poisson=l1 == 0.0,
                                             nfields=c.get("fields", 1), **kw)


_held = {}


def _setup(c):
    key = json.dumps({k: v for k, v in c.items() if k != "name"}, sort_keys=True)
    if key not in _held:
        _held.clear()
        _held[key] = _Setup(c)
    return _held[key]


def _field(s, gen, masked=False, n=1):
    """Random nodal values that agree on shared nodes; zero on the Dirichlet boundary if masked."""
    v = torch.rand((n, int(s.mesh.gid.max()) + 1), generator=gen, device="cuda", dtype=torch.float64) * 2 - 1
    out = v[:, s.gid]
    if masked:
        out[:, _boundary(s.mesh)] = 0
    return out.reshape(-1)


def _boundary(m):
    """Dirichlet nodes: the outer faces of the box."""
    Nq = m.N + 1
    b = torch.zeros((m.nz, m.ny, m.nx, Nq, Nq, Nq), dtype=torch.bool, device="cuda")
    b[0, :, :, 0], b[-1, :, :, -1] = True, True
    b[:, 0, :, :, 0], b[:, -1, :, :, -1] = True, True
    b[:, :, 0, :, :, 0], b[:, :, -1, :, :, -1] = True, True
    return b.reshape(-1)


def _modes(m, gen):
    """A smooth load at the nodes: sine modes with random amplitudes."""
    a = (torch.rand((3, 3, 3), generator=gen, device="cuda", dtype=torch.float64) * 2 - 1).tolist()
    a[0][0][0] = 2.0
    s = [[torch.sin((k + 1) * math.pi * torch.from_numpy(x).cuda()) for k in range(3)] for x in (m.x, m.y, m.z)]
    return 3 * math.pi ** 2 * sum(a[i][j][k] * s[0][i] * s[1][j] * s[2][k]
                                  for i in range(3) for j in range(3) for k in range(3))


def prepare(c, seed):
    s = _setup(c)
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    op, L = c["op"], s.L
    st = {"op": op, "setup": s}
    if op == "operator":
        st["q"] = _field(s, gen, n=c["fields"])
        st["Aq"] = torch.empty_like(st["q"])
    elif op == "average":
        dt = torch.float64 if c["dtype"] == "f64" else torch.float32
        st["u"] = (torch.rand((c["nvec"], L), generator=gen, device="cuda", dtype=torch.float64) * 2 - 1).to(dt)
        st["v"] = torch.empty_like(st["u"])
        st["nvec"] = c["nvec"]
    elif op == "rhs":
        for k in ("Ue", "U", "BF"):
            st[k] = _field(s, gen, n=3)
        st["mue"], st["irho"] = 1.0 + 0.5 * _field(s, gen), 1.0 + 0.25 * _field(s, gen)
        st["div"] = _field(s, gen)
        st["rhs"] = torch.empty(L, dtype=torch.float64, device="cuda")
    elif op == "smoother":
        st["r"] = _field(s, gen, masked=True).float()
        st["z"] = torch.empty_like(st["r"])
    elif op == "vcycle":
        st["r"] = _field(s, gen, masked=True)
        st["z"] = torch.empty_like(st["r"])
    else:
        st["f"] = _modes(s.mesh, gen)
        st["b"], st["x"] = torch.empty_like(st["f"]), torch.empty_like(st["f"])
    return st


G0 = 150.0   # bd0 / dt of the pressure right-hand side


def run(st):
    op, h = st["op"], st["setup"].handle
    if op == "operator":
        h.operator(st["q"], st["Aq"])
        return st["Aq"]
    if op == "average":
        torch.mul(st["u"], st["setup"].weight, out=st["v"])
        h.gather_scatter(st["v"], "add", nvec=st["nvec"])
        return st["v"]
    if op == "rhs":
        return h.compute(st["Ue"], st["U"], st["BF"], st["mue"], st["irho"], st["div"], G0, rhs=st["rhs"])
    if op == "smoother":
        h.mg_smoother(0, st["r"], st["z"])
        return st["z"]
    if op == "vcycle":
        h.preconditioner(st["r"], st["z"])
        return st["z"]
    st["b"].copy_(st["f"])      # the solve leaves its residual in b
    st["x"].zero_()
    h.solve(st["b"], st["x"])
    return st["x"]


def work(c):
    """Vectors in and out once, and what the element keeps (geometric factors of
    the general operator, 1D operators of the box solves); iterative solves are
    counted as one iteration, since how many they need is not known beforehand."""
    N, E = c["N"], c["nx"] * c["ny"] * c["nz"]
    Nq, nl = N + 1, N + 3
    L = E * Nq ** 3
    ax = (12 * Nq + 20) * L
    op = c["op"]
    if op == "operator":
        f = c["fields"]
        return {"bytes": 8 * L * (2 * f + (6 if c["lambda1"] == 0.0 else 7)), "flops": f * ax}
    if op == "average":
        w = 8 if c["dtype"] == "f64" else 4
        return {"bytes": w * L * (2 * c["nvec"] + 1), "flops": 2 * L * c["nvec"]}
    if op == "rhs":     # Ue, BF, mue, irho, div in, rhs out, corners; two curls, a gradient, a divergence
        return {"bytes": L * 8 * 10 + E * 192, "flops": L * (26 * 2 * Nq + 250)}
    box = 12 * nl ** 4 * E
    ops = E * 3 * nl * nl * (2 if c.get("options") == "mixed-asm-bf16" else 4)
    if op == "smoother":
        return {"bytes": 8 * L + ops, "flops": box}
    if c["options"] == "jacobi":
        return {"bytes": 64 * L, "flops": ax}
    if c["options"] == "fp64-chebyshev":
        return {"bytes": 16 * L, "flops": 4 * ax}
    return {"bytes": 16 * L + ops + (64 * L if op == "solve" else 0), "flops": 6 * (ax + box)}


def tolerance(c):
    """About four times what two correct evaluations were measured to differ by:
    run() and exact(), or a V-cycle with its level operators' geometric factors
    stored and formed from the element corners."""
    op = c["op"]
    if op == "operator":      # up to 3.5e-12: the factors are differences of close coordinates
        return {"rel": 1.5e-11}
    if op == "rhs":           # 5.2e-13
        return {"rel": 2e-12}
    if op == "average":       # a handful of terms
        return {"rel": 1e-15 if c["dtype"] == "f64" else 3e-7}
    if op == "smoother":      # 1.3e-7 in FP32; 3.8e-3 with BF16 operands
        return {"rel": 6e-7} if c["options"] == "mixed-ras" else {"rel": 1.5e-2}
    if op == "vcycle":        # 2.3e-14, 4.2e-7, and 2.5e-4 where roundings to BF16 flip
        return {"rel": {"fp64-chebyshev": 1e-13, "mixed-ras": 2e-6, "mixed-asm-bf16": 1e-3}[c["options"]]}
    return {"rel": 3e-9}      # up to 6.7e-10: a solve stops at 1e-8 of its first residual


# ------------------------------------------------------------------ 64-bit results in plain torch

def _gll(N):
    """Gauss-Lobatto-Legendre nodes, weights and the derivative matrix D[i][j] = l_j'(z_i)."""
    P = np.polynomial.legendre.Legendre.basis(N)
    z = np.concatenate([[-1.0], np.sort(np.real(P.deriv().roots())), [1.0]])
    for _ in range(4):      # polish the inner roots
        z[1:-1] -= P.deriv()(z[1:-1]) / P.deriv(2)(z[1:-1])
    w = 2.0 / (N * (N + 1) * P(z) ** 2)
    p = P(z)
    D = np.zeros((N + 1, N + 1))
    for i in range(N + 1):
        for j in range(N + 1):
            if i != j:
                D[i, j] = p[i] / (p[j] * (z[i] - z[j]))
    D[0, 0], D[N, N] = -N * (N + 1) / 4.0, N * (N + 1) / 4.0
    return z, w, torch.from_numpy(D).cuda()


def _d(D, u):
    """Derivatives in r, s, t of u[E][k][j][i]."""
    E, n = u.shape[0], D.shape[0]
    return u @ D.T, D @ u, (D @ u.reshape(E, n, n * n)).reshape(u.shape)


class _Geometry:
    def __init__(self, m):
        Nq = m.N + 1
        z, w, self.D = _gll(m.N)
        self.shape = (m.E, Nq, Nq, Nq)
        w = torch.from_numpy(w).cuda()
        W = w[:, None, None] * w[None, :, None] * w[None, None, :]
        x, y, zz = (torch.from_numpy(a).cuda().reshape(self.shape) for a in (m.x, m.y, m.z))
        (xr, xs, xt), (yr, ys, yt), (zr, zs, zt) = (_d(self.D, a) for a in (x, y, zz))
        J = xr * (ys * zt - zs * yt) - yr * (xs * zt - zs * xt) + zr * (xs * yt - ys * xt)
        self.r = [(ys * zt - zs * yt) / J, (zs * xt - xs * zt) / J, (xs * yt - ys * xt) / J]
        self.s = [(zr * yt - yr * zt) / J, (xr * zt - zr * xt) / J, (yr * xt - xr * yt) / J]
        self.t = [(yr * zs - zr * ys) / J, (zr * xs - xr * zs) / J, (xr * ys - yr * xs) / J]
        self.J, self.JW, self.w = J, J * W, w
        self.gid = torch.from_numpy(m.gid).cuda()
        self.count = int(m.gid.max()) + 1

    def sum(self, v):
        """Sum over the copies of each node."""
        t = torch.zeros(self.count, dtype=v.dtype, device=v.device)
        return t.index_add_(0, self.gid, v.reshape(-1))[self.gid].reshape(v.shape)

    def grad(self, u):
        a, b, c = _d(self.D, u)
        return [self.r[q] * a + self.s[q] * b + self.t[q] * c for q in range(3)]

    def weak(self, f):
        """Sum over directions of the transposed derivative of JW (grad r_d . f)."""
        E, n = self.shape[0], self.D.shape[0]
        a, b, c = (self.JW * (g[0] * f[0] + g[1] * f[1] + g[2] * f[2]) for g in (self.r, self.s, self.t))
        return a @ self.D + self.D.T @ b + (self.D.T @ c.reshape(E, n, n * n)).reshape(self.shape)

    def ax(self, q, lambda1):
        out = self.weak(self.grad(q))
        return out + lambda1 * self.JW * q if lambda1 else out


def _exact_operator(c, s, st):
    g = _Geometry(s.mesh)
    mask = _boundary(s.mesh).reshape(g.shape)
    return torch.cat([g.sum(g.ax(q.reshape(g.shape), c["lambda1"]).masked_fill(mask, 0.0)).reshape(-1)
                      for q in st["q"].reshape(c["fields"], -1)])


def _exact_average(c, s, st):
    gid, n = s.gid, int(s.mesh.gid.max()) + 1
    deg = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(
        0, gid, torch.ones(s.L, dtype=torch.float64, device="cuda"))
    return torch.stack([torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, gid, u.double())[gid] / deg[gid]
                        for u in st["u"]])


def _exact_rhs(s, st):
    g = _Geometry(s.mesh)
    lmm = g.sum(g.JW)
    vec = lambda k: [a.reshape(g.shape) for a in st[k].reshape(3, -1)]     # noqa: E731
    mue, irho, div = (st[k].reshape(g.shape) for k in ("mue", "irho", "div"))

    def curl(f):
        u, v, w = (g.grad(a) for a in f)
        return [w[1] - v[2], u[2] - w[0], v[0] - u[1]]
    W = [g.sum(g.JW * a) / lmm for a in curl(vec("Ue"))]
    nu, gd = mue * irho, g.grad(div)
    F = [g.sum(b - nu * g.JW * (a - 4.0 / 3.0 * d)) / lmm for a, b, d in zip(curl(W), vec("BF"), gd)]
    out = g.weak(F) + G0 * g.JW * div
    # inflow faces take the velocity's flux, symmetry faces that of F
    bc, U = torch.from_numpy(s.bc).cuda().reshape(-1, 6), vec("U")
    last = s.mesh.N
    faces = [(0, (slice(None), 0), g.t, -1), (5, (slice(None), last), g.t, 1),
             (1, (slice(None), slice(None), 0), g.s, -1), (3, (slice(None), slice(None), last), g.s, 1),
             (2, (slice(None),) * 3 + (last,), g.r, 1), (4, (slice(None),) * 3 + (0,), g.r, -1)]
    for f, at, d, sign in faces:
        n = [sign * a[at] for a in d]      # the unit normal times the surface factor is n J w w
        ww = g.J[at] * g.w[:, None] * g.w[None, :]
        kind = bc[:, f][:, None, None]
        inflow = G0 * sum(a * b[at] for a, b in zip(n, U))
        symmetry = sum(a * b[at] for a, b in zip(n, F))
        out[at] -= ww * torch.where(kind == 3, inflow, torch.where(kind == 7, symmetry, torch.zeros_like(inflow)))
    return out.reshape(-1)


def _exact_smoother(c, s, st):
    """The overlapping Schwarz smoother: on each element extended by one layer of
    each face neighbour's nodes, the inverse of the separable Helmholtz operator
    of a brick of the element's mean lengths."""
    m, N = s.mesh, c["N"]
    Nq, nl, E = N + 1, N + 3, m.E
    _, w, D = _gll(N)
    D = D.cpu()
    wt = torch.from_numpy(w)
    xyz = torch.stack([torch.from_numpy(a).reshape(m.nz, m.ny, m.nx, Nq, Nq, Nq) for a in (m.x, m.y, m.z)])
    axes = (2, 1, 0)          # element axis and box axis of r, s, t
    inner = wt[:N - 1][:, None] * wt[:N - 1][None, :]
    A0 = D.T @ (wt[:, None] * D)
    S, lam = [], []
    for d in range(3):
        ax = 4 + axes[d]
        span = xyz.select(ax, Nq - 1) - xyz.select(ax, 0)
        span = (span ** 2).sum(0)[..., 1:Nq - 1, 1:Nq - 1]
        mid = 1.0 / torch.sqrt((inner / span).sum((-1, -2)) / inner.sum())     # [nz][ny][nx]
        e = axes[d]
        n = mid.shape[e]
        left, right = mid.clone(), mid.clone()
        left.narrow(e, 1, n - 1).copy_(mid.narrow(e, 0, n - 1))
        right.narrow(e, 0, n - 1).copy_(mid.narrow(e, 1, n - 1))
        shape = [1, 1, 1]
        shape[e] = n
        at = torch.arange(n).reshape(shape).expand(mid.shape).reshape(-1)
        lo, hi = at == 0, at == n - 1
        a, b = torch.zeros(E, nl, nl, dtype=torch.float64), torch.zeros(E, nl, dtype=torch.float64)
        lm, ll, lr = mid.reshape(-1), left.reshape(-1), right.reshape(-1)
        a[:, 1:N + 2, 1:N + 2] = 2.0 / lm[:, None, None] * A0
        b[:, 1:N + 2] = 0.5 * lm[:, None] * wt
        # Dirichlet ends: the end node is cut off (its rows and columns become the identity's)
        for cut, node, ghost in ((lo, 1, 0), (hi, N + 1, N + 2)):
            a[cut, node, :], a[cut, :, node] = 0.0, 0.0
            a[cut, node, node], a[cut, ghost, ghost] = 1.0, 1.0
            b[cut, node], b[cut, ghost] = 1.0, 1.0
        for join, node, ghost, h, p, q in ((~lo, 1, 0, ll, N, N - 1), (~hi, N + 1, N + 2, lr, 0, 1)):
            f = 2.0 / h[join]
            a[join, ghost, ghost] = f * A0[q, q]
            a[join, node, ghost], a[join, ghost, node] = f * A0[p, q], f * A0[p, q]
            a[join, node, node] += f * A0[p, p]
            b[join, ghost] = 0.5 * h[join] * wt[q]
            b[join, node] += 0.5 * h[join] * wt[p]
        r = b.rsqrt()
        val, vec = torch.linalg.eigh(r[:, :, None] * a * r[:, None, :])
        vec = r[:, :, None] * vec
        vec[lo, :2], vec[hi, nl - 2:] = 0.0, 0.0
        S.append(vec.cuda())
        lam.append(val.cuda())
    total = lam[2][:, :, None, None] + lam[1][:, None, :, None] + lam[0][:, None, None, :]
    inv = torch.where(total > 1e-5, 1.0 / (total + c["lambda1"]), torch.zeros_like(total))

    box = torch.zeros(m.nz, m.ny, m.nx, nl, nl, nl, dtype=torch.float64, device="cuda")
    u = st["r"].double().reshape(m.nz, m.ny, m.nx, Nq, Nq, Nq)
    box[..., 1:-1, 1:-1, 1:-1] = u
    k = slice(1, -1)
    box[1:, :, :, 0, k, k], box[:-1, :, :, -1, k, k] = u[:-1, :, :, N - 1], u[1:, :, :, 1]
    box[:, 1:, :, k, 0, k], box[:, :-1, :, k, -1, k] = u[:, :-1, :, :, N - 1], u[:, 1:, :, :, 1]
    box[:, :, 1:, k, k, 0], box[:, :, :-1, k, k, -1] = u[:, :, :-1, :, :, N - 1], u[:, :, 1:, :, :, 1]
    v = box.reshape(E, nl, nl, nl)

    def both(v, Sx, Sy, Sz):        # apply a matrix to each axis: v[k][j][i] -> i by Sx, j by Sy, k by Sz
        v = v @ Sx.transpose(1, 2).contiguous()[:, None]
        v = Sy[:, None] @ v
        return (Sz @ v.reshape(E, nl, nl * nl)).reshape(v.shape)
    T = [a.transpose(1, 2).contiguous() for a in S]
    v = both(both(v, *T) * inv, *S).reshape(box.shape)
    z = v[..., k, k, k].clone()
    g = torch.from_numpy(m.gid).cuda()
    mask = _boundary(m)

    def summed(a):
        a = a.reshape(-1).masked_fill(mask, 0.0)
        return torch.zeros(int(m.gid.max()) + 1, dtype=a.dtype, device="cuda").index_add_(0, g, a)[g]
    ones = torch.ones_like(u)
    if "ras" in c["options"]:
        deg = summed(ones)
        return summed(z.reshape(-1) / deg.clamp(min=1.0))
    # additive: what each neighbour's box found on its ghost layer is added to the layer it came from
    for t, ov in ((z, v), (ones, torch.ones_like(v))):
        t[:-1, :, :, N - 1] += ov[1:, :, :, 0, k, k]
        t[1:, :, :, 1] += ov[:-1, :, :, -1, k, k]
        t[:, :-1, :, :, N - 1] += ov[:, 1:, :, k, 0, k]
        t[:, 1:, :, :, 1] += ov[:, :-1, :, k, -1, k]
        t[:, :, :-1, :, :, N - 1] += ov[:, :, 1:, k, k, 0]
        t[:, :, 1:, :, :, 1] += ov[:, :, :-1, k, k, -1]
    deg = summed(ones)
    return summed(z.reshape(-1) / deg.clamp(min=1.0))


def _exact_solve(c, s, st):
    """The solution of the assembled system, by CG with the operator's diagonal, to 1e-12."""
    g = _Geometry(s.mesh)
    mask = _boundary(s.mesh).reshape(g.shape)
    D2 = g.D ** 2
    E, n = g.shape[0], g.D.shape[0]
    G = lambda a, b: g.JW * (a[0] * b[0] + a[1] * b[1] + a[2] * b[2])      # noqa: E731
    dd = torch.diagonal(g.D)
    diag = G(g.r, g.r) @ D2 + D2.T @ G(g.s, g.s) + (D2.T @ G(g.t, g.t).reshape(E, n, n * n)).reshape(g.shape)
    diag = diag + 2 * (G(g.r, g.s) * dd[None, None, None, :] * dd[None, None, :, None] +
                       G(g.r, g.t) * dd[None, None, None, :] * dd[None, :, None, None] +
                       G(g.s, g.t) * dd[None, None, :, None] * dd[None, :, None, None])
    minv = 1.0 / g.sum(diag + c["lambda1"] * g.JW)
    keep = (~mask).double()
    wgt = keep / g.sum(torch.ones_like(keep))
    A = lambda v: g.sum(g.ax(v, c["lambda1"])) * keep                        # noqa: E731
    r = g.sum(st["f"].reshape(g.shape)) * keep
    x, p, rz = torch.zeros_like(r), None, 0.0
    goal = 1e-12 * math.sqrt(float((wgt * r * r).sum()))
    for it in range(6000):
        z = minv * r
        new = (wgt * r * z).sum()
        p = z if p is None else z + (new / rz) * p
        rz = new
        Ap = A(p)
        a = rz / (wgt * p * Ap).sum()
        x += a * p
        r -= a * Ap
        if it % 50 == 49 and math.sqrt(float((wgt * r * r).sum())) < goal:
            break
    return x.reshape(-1)


def exact(c, seed):
    op = c["op"]
    if op == "vcycle":        # a V-cycle's value hangs on its own AMG hierarchy and eigenvalue bounds
        return None
    s = _setup(c)
    st = prepare(c, seed)
    if op == "operator":
        return _exact_operator(c, s, st)
    if op == "average":
        return _exact_average(c, s, st)
    if op == "rhs":
        return _exact_rhs(s, st)
    if op == "smoother":
        return _exact_smoother(c, s, st)
    return _exact_solve(c, s, st)
