"""Performance cases of the vertex-patch Schwarz smoother library.

A case is one call of a public entry point, as a multigrid program makes it:

  operator   Level.vmult            the SIPG operator of the outer CG
  residual   Level.residual         b - A x before a restriction
  additive   SchwarzPreconditioner.vmult, all patches at once
  sweep      SchwarzSmoother.vmult, one multiplicative sweep over the red-black
             colors from a zero guess (the pre-smoother of a V-cycle)
  solve      GMGSolver.solve, GMG-preconditioned CG to 1e-8

on a Cartesian Poisson mesh ("cartesian"), a Poisson mesh with moved interior
vertices ("moved") or a Cartesian linear elasticity level ("elastic"), with FP64
or FP32 level vectors and patch solves.  Right-hand sides are random, uniform in
[-1, 1], as in the reference's smoother benchmarks.
"""
import numpy as np
import torch

import tpss_amd as t

MU, LAMBDA = 1.0, 10.0
#: penalty factors of the three meshes
IP = {"cartesian": 1.0, "moved": 4.0, "elastic": 10.0}
#: vertex movement of the moved meshes in cell lengths
AMPLITUDE = 0.15
#: V-cycles of a 1e-8 solve on a Cartesian Poisson mesh
SOLVE_CYCLES = 4
SOLVE_TOL = 1e-8


def _case(name, call, mesh, dim, degree, n, precision, relaxation=1.0, levels=0):
    c = {"call": call, "mesh": mesh, "dim": dim, "degree": degree, "n": n, "precision": precision,
         "relaxation": relaxation, "levels": levels}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a coarse level of a 2D V-cycle: 4096 DoFs, eight color launches, latency only
        _case("sweep_2d_q3_16_f64", "sweep", "cartesian", 2, 3, 16, "f64"),
        # one additive smoothing step of the 2D model problem (128 x 128 cells)
        _case("additive_2d_q3_128_f64", "additive", "cartesian", 2, 3, 128, "f64", 0.25),
        # the residual before a restriction on a level of odd size, low degree
        _case("residual_3d_q2_33_f64", "residual", "cartesian", 3, 2, 33, "f64"),
        # a middle level of the mixed-precision V-cycle
        _case("sweep_3d_q3_16_f32", "sweep", "cartesian", 3, 3, 16, "f32"),
        # a sweep of the highest degree on a level of odd size
        _case("sweep_3d_q4_27_f64", "sweep", "cartesian", 3, 4, 27, "f64"),
        # the fine level of the 3D model problem (16.8M DoFs): FP64 smoother
        _case("sweep_3d_q3_64_f64", "sweep", "cartesian", 3, 3, 64, "f64"),
        # the same level in the mixed-precision V-cycle
        _case("sweep_3d_q3_64_f32", "sweep", "cartesian", 3, 3, 64, "f32"),
        # additive smoother with FP32 applies on a mesh with moved vertices, Q4
        _case("additive_moved_3d_q4_48_f32", "additive", "moved", 3, 4, 48, "f32", 0.7),
        # the outer CG's FP64 operator on the mesh with moved vertices
        _case("operator_moved_3d_q3_64_f64", "operator", "moved", 3, 3, 64, "f64"),
        # the damped multiplicative smoother of the mixed V-cycle on moved vertices
        _case("sweep_moved_3d_q3_40_f32", "sweep", "moved", 3, 3, 40, "f32", 0.7),
        # the linear elasticity smoother of the mixed V-cycle (21.2M DoFs)
        _case("sweep_elastic_3d_q2_64_f32", "sweep", "elastic", 3, 2, 64, "f32"),
        # a whole solve: mixed-precision GMG-CG to 1e-8, six levels down to 2^3 cells
        _case("solve_3d_q3_64_f32", "solve", "cartesian", 3, 3, 64, "f32", 1.0, 6),
    ]


#: largest vectors (DoFs) drawn per call and mesh: no drawn case costs more than
#: the largest listed one
_LARGEST = {("operator", "cartesian"): 2 ** 24, ("residual", "cartesian"): 2 ** 24,
            ("additive", "cartesian"): 2 ** 24, ("sweep", "cartesian"): 2 ** 24,
            ("operator", "moved"): 2 ** 24, ("residual", "moved"): 2 ** 24,
            ("additive", "moved"): 1.2e7, ("sweep", "moved"): 4.0e6,
            ("operator", "elastic"): 2e7, ("residual", "elastic"): 2e7,
            ("additive", "elastic"): 2e7, ("sweep", "elastic"): 1e7}


def draw(rng):
    call = rng.choice(["operator", "residual", "additive", "sweep", "sweep", "sweep", "solve"])
    dim = rng.choice([2, 3, 3])
    degree = rng.choice([1, 2, 2, 3, 3, 3, 4])
    precision = rng.choice(["f64", "f32"])
    if call == "solve":
        degree = rng.choice([2, 3, 3])
        levels = rng.randint(3, 5)
        coarse = rng.choice([2, 3])
        return _case("", call, "cartesian", dim, degree, coarse << (levels - 1), precision, 1.0,
                     levels)
    mesh = rng.choice(["cartesian", "moved", "elastic"])
    n_comp = dim if mesh == "elastic" else 1
    largest = _LARGEST[(call, mesh)] if dim == 3 else 2e6
    dofs = np.exp(rng.uniform(np.log(4e3), np.log(largest)))
    n = int((dofs / (n_comp * (degree + 1) ** dim)) ** (1.0 / dim))
    n = max(4, min(n, 128 if dim == 3 else 700))
    relaxation = {"additive": {2: 0.25, 3: 0.15}[dim], "sweep": 0.7 if mesh == "moved" else 1.0}
    return _case("", call, mesh, dim, degree, n, precision, relaxation.get(call, 1.0))


def _n_dofs(case):
    n_comp = case["dim"] if case["mesh"] == "elastic" else 1
    return n_comp * (case["n"] * (case["degree"] + 1)) ** case["dim"]


def _vertices(case, seed):
    """(n+1)^dim vertices, x fastest, the interior ones moved by up to AMPLITUDE h"""
    if case["mesh"] != "moved":
        return None
    dim, n = case["dim"], case["n"]
    g = np.arange(n + 1) / n
    v = np.stack(np.meshgrid(*[g] * dim, indexing="ij")[::-1], axis=-1)
    inner = (slice(1, n),) * dim
    noise = np.random.default_rng(seed).uniform(-1.0, 1.0, v[inner].shape)
    v[inner] += AMPLITUDE / n * noise
    return v.reshape(-1, dim)


def _rhs(case, seed, dtype, device="cuda"):
    """random level vectors: the right-hand side, and the x of a residual"""
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    return [torch.rand(_n_dofs(case), generator=g, device=device, dtype=dtype) * 2 - 1
            for _ in range(2 if case["call"] == "residual" else 1)]


def _dtype(case):
    # the outer CG of a solve keeps its vectors in FP64
    return torch.float32 if case["precision"] == "f32" and case["call"] != "solve" else torch.float64


def prepare(case, seed):
    dim, degree, n, call = case["dim"], case["degree"], case["n"], case["call"]
    prec = t.F32 if case["precision"] == "f32" else t.F64
    ip = IP[case["mesh"]]
    state = {"call": call, "rhs": _rhs(case, seed, _dtype(case))}
    state["out"] = torch.empty_like(state["rhs"][0])
    if call == "solve":
        levels = case["levels"]
        state["solver"] = t.GMGSolver(dim, degree, n >> (levels - 1), levels, ip_factor=ip,
                                      mg_precision=prec, relaxation=case["relaxation"])
        return state
    state["level"] = t.Level(dim, degree, n, ip_factor=ip, vertices=_vertices(case, seed),
                             precision=prec,
                             elasticity=(MU, LAMBDA) if case["mesh"] == "elastic" else None)
    if call == "additive":
        state["smoother"] = t.SchwarzPreconditioner(state["level"], t.ADDITIVE,
                                                    relaxation=case["relaxation"])
    elif call == "sweep":
        state["smoother"] = t.SchwarzSmoother(state["level"], t.MULTIPLICATIVE,
                                              relaxation=case["relaxation"])
    return state


def run(state):
    call, out, rhs = state["call"], state["out"], state["rhs"]
    if call == "operator":
        state["level"].vmult(out, rhs[0])
    elif call == "residual":
        state["level"].residual(out, rhs[0], rhs[1])
    elif call == "solve":
        state["solver"].solve(out, rhs[0], rel_tol=SOLVE_TOL)
    else:
        state["smoother"].vmult(out, rhs[0])
    return out


def work(case):
    """compulsory bytes: inputs read once, outputs written once (and the vertices
    of a moved mesh); operations: the operator's and the patch solves' one
    direction at a time contractions, without geometry"""
    dim, np1, n, call = case["dim"], case["degree"] + 1, case["n"], case["call"]
    n_comp = dim if case["mesh"] == "elastic" else 1
    N = _n_dofs(case)
    size = 4 if _dtype(case) == torch.float32 else 8
    nbytes = (3 if call == "residual" else 2) * N * size
    if case["mesh"] == "moved":
        nbytes += dim * (n + 1) ** dim * 8
    # 1D contractions per DoF: dim line operators over three cells and the masses
    apply = N * 2 * np1 * (3 * dim + (5 if dim == 3 else 2))
    K = 2 * np1
    patches = n_comp * (n - 1) ** dim * (4 * dim * K ** (dim + 1) + 2 * K ** dim)
    flops = {"operator": apply, "residual": apply + N, "additive": patches,
             "sweep": patches + 2 ** dim * apply}.get(call)
    if call == "solve":
        # every cycle: two sweeps and a residual on a geometric series of levels,
        # and the operator of the outer CG
        levels = 2 ** dim / (2 ** dim - 1)
        flops = SOLVE_CYCLES * (levels * (2 * (patches + 2 ** dim * apply) + apply) + apply)
    return {"bytes": int(nbytes), "flops": int(flops)}


# ---------------------------------------------------------------------------
# The same results in 64 bits with plain torch and numpy.  Fields live on the
# cells as [component][cells: z, y, x][nodes: z, y, x]; axis d of the mesh is
# the d-th from the end of either group.
# ---------------------------------------------------------------------------

class _Basis:
    """Lagrange basis on Gauss-Lobatto nodes of [0, 1], tabulated at Gauss points"""

    def __init__(self, p):
        leg = np.polynomial.legendre
        c = np.zeros(p + 1)
        c[p] = 1.0
        inner = leg.legroots(leg.legder(c)) if p > 1 else np.zeros(0)
        self.nodes = 0.5 + 0.5 * np.concatenate([[-1.0], inner, [1.0]])
        self.lobatto_w = 1.0 / (p * (p + 1) * leg.legval(2 * self.nodes - 1, c) ** 2)
        x, w = leg.leggauss(p + 1)
        self.qx, self.qw = 0.5 + 0.5 * x, 0.5 * w
        self.V, self.D = self.table(self.qx)  # [point, node]
        self.fv, self.fd = self.table(np.array([0.0, 1.0]))

    def table(self, x):
        z = self.nodes
        m = len(z)
        V, D = np.ones((len(x), m)), np.zeros((len(x), m))
        for j in range(m):
            for k in range(m):
                if k != j:
                    D[:, j] = (D[:, j] * (x - z[k]) + V[:, j]) / (z[j] - z[k])
                    V[:, j] = V[:, j] * (x - z[k]) / (z[j] - z[k])
        return V, D


def _line_matrices(b, h, left, right, ip, cons, pen):
    """1D mass and SIPG matrix of a line of cells of lengths h [..., cells];
    left / right [...]: the line's ends are physical boundaries (cut faces keep
    their own cell's half of the interior face terms otherwise)"""
    m, cells = len(b.nodes), h.shape[-1]
    gamma = (m - 1) * m
    M = np.zeros(h.shape[:-1] + (cells * m,) * 2)
    L = np.zeros_like(M)
    mass, stiff = (b.V.T * b.qw) @ b.V, (b.D.T * b.qw) @ b.D
    for c in range(cells):
        hc, at = h[..., c, None, None], slice(c * m, c * m + m)
        M[..., at, at] += hc * mass
        L[..., at, at] += cons * stiff / hc
        for f in (0, 1):
            bound = (left if f == 0 else right) if c == (0 if f == 0 else cells - 1) else False
            a = np.where(bound, 1.0, 0.5)[..., None, None]
            nrm, v, g = 2 * f - 1, b.fv[f][:, None], b.fd[f][:, None] / hc
            sigma = ip * a * 2 * gamma / hc
            gT = np.swapaxes(g, -1, -2)
            L[..., at, at] += -cons * a * nrm * (v * gT + g * v.T) + pen * sigma * v * v.T
    for c in range(cells - 1):
        h0, h1 = h[..., c, None, None], h[..., c + 1, None, None]
        sigma = ip * gamma * (0.5 / h0 + 0.5 / h1)
        lo, hi = slice(c * m, c * m + m), slice(c * m + m, c * m + 2 * m)
        v0, v1 = b.fv[1][:, None], b.fv[0][:, None]
        g0, g1 = b.fd[1][:, None] / h0, b.fd[0][:, None] / h1
        block = -cons * 0.5 * (v0 * np.swapaxes(g1, -1, -2) - g0 * v1.T) - pen * sigma * v0 * v1.T
        L[..., lo, hi] += block
        L[..., hi, lo] += np.swapaxes(block, -1, -2)
    return M, L


def _derivative_matrices(b, n):
    """1D matrices of the mixed elasticity terms on n cells of length 1/n:
    G = int phi_i phi_j' and S = -sum over faces of [phi_i] {phi_j}"""
    m = len(b.nodes)
    G, S = np.zeros((n * m, n * m)), np.zeros((n * m, n * m))
    g = (b.V.T * b.qw) @ b.D
    for c in range(n):
        at = slice(c * m, c * m + m)
        G[at, at] = g
        for f in (0, 1):
            nrm, nb = 2 * f - 1, c + 2 * f - 1
            if 0 <= nb < n:
                S[at, at] -= 0.5 * nrm * np.outer(b.fv[f], b.fv[f])
                S[at, nb * m:nb * m + m] -= 0.5 * nrm * np.outer(b.fv[f], b.fv[1 - f])
            else:
                S[at, at] -= nrm * np.outer(b.fv[f], b.fv[f])
    return G, S


def _to_grid(x, dim, n, m):
    """[comp][cells][nodes] -> [comp][grid points z, y, x]"""
    x = x.reshape((-1,) + (n,) * dim + (m,) * dim)
    order = [0]
    for d in range(dim):
        order += [1 + d, 1 + dim + d]
    return x.permute(order).reshape((-1,) + (n * m,) * dim)


def _from_grid(x, dim, n, m):
    x = x.reshape((-1,) + (n, m) * dim)
    return x.permute([0] + [1 + 2 * d for d in range(dim)] + [2 + 2 * d for d in range(dim)])


def _along(A, x, axis):
    """y = A x along one axis"""
    return torch.movedim(torch.tensordot(x, A, dims=([axis], [1])), -1, axis)


class _KroneckerOperator:
    """Poisson / elasticity on a uniform Cartesian mesh: sums of Kronecker products
    of 1D matrices over the whole line of n cells"""

    def __init__(self, case, b, device):
        n, self.dim = case["n"], case["dim"]
        self.elastic = case["mesh"] == "elastic"
        self.n, self.m = n, len(b.nodes)
        h, ip = np.full(n, 1.0 / n), IP[case["mesh"]]
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)  # noqa: E731
        line = lambda cons, pen: dev(_line_matrices(b, h, True, True, ip, cons, pen)[1])  # noqa: E731
        self.M = dev(_line_matrices(b, h, True, True, ip, 1.0, 1.0)[0])
        if self.elastic:
            self.L = {True: line(2 * MU + LAMBDA, 2 * MU + LAMBDA), False: line(MU, 2 * MU)}
            G, S = _derivative_matrices(b, n)
            self.G, self.Gt, self.S, self.St = dev(G), dev(G.T), dev(S), dev(S.T)
        else:
            self.L = {False: line(1.0, 1.0)}

    def apply(self, x):
        g = _to_grid(x, self.dim, self.n, self.m)
        y = torch.zeros_like(g)
        dims = range(self.dim)
        for c in range(g.shape[0]):
            for d in dims:
                v = _along(self.L[self.elastic and c == d], g[c], self.dim - 1 - d)
                for e in dims:
                    if e != d:
                        v = _along(self.M, v, self.dim - 1 - e)
                y[c] += v
            for a in dims if self.elastic else ():
                if a == c:
                    continue
                # test component a, trial component c
                u = g[c]
                for e in dims:
                    if e not in (a, c):
                        u = _along(self.M, u, self.dim - 1 - e)
                two = lambda A, C: _along(C, _along(A, u, self.dim - 1 - a), self.dim - 1 - c)  # noqa: E731
                y[a] += MU * (two(self.G + self.St, self.Gt) + two(self.G, self.S))
                y[a] += LAMBDA * (two(self.Gt + self.S, self.G) + two(self.Gt, self.St))
        return _from_grid(y, self.dim, self.n, self.m).reshape(-1)


class _MovedOperator:
    """Poisson on multilinear cells: QGauss(p+1) on cells and faces"""

    def __init__(self, case, b, vertices, device):
        self.b, self.dim, self.n, self.m = b, case["dim"], case["n"], len(b.nodes)
        self.ip, self.gamma = IP[case["mesh"]], (self.m - 1) * self.m
        self.dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(device)
        self.V, self.D = self.dev(b.V), self.dev(b.D)
        n, dim = self.n, self.dim
        v = self.dev(vertices).reshape((n + 1,) * dim + (dim,))
        # corners as a multilinear "nodal" field [dim][cells][2, 2, 2]
        for d in range(dim):
            v = v.unfold(d, 2, 1)
        self.corner = torch.movedim(v, dim, 0)

    def _axis(self, d, nodes=True):
        """position of mesh direction d in [cells][nodes]"""
        return (2 if nodes else 1) * self.dim - 1 - d

    def _jacobian(self, x):
        """columns J[b] = [a][cells][points] at the tensor points x[d]"""
        cols = []
        for e in range(self.dim):
            v = self.corner
            for d in range(self.dim):
                t1 = np.stack([-np.ones_like(x[d]), np.ones_like(x[d])], 1) if d == e else \
                    np.stack([1 - x[d], x[d]], 1)
                v = _along(self.dev(t1), v, 1 + self._axis(d))
            cols.append(v)
        return torch.stack(cols, 1)  # [a][b][cells][points]

    @staticmethod
    def _inverse(J):
        """inverse (rows b, columns a) and determinant of J[a][b]"""
        if J.shape[0] == 2:
            det = J[0, 0] * J[1, 1] - J[0, 1] * J[1, 0]
            rows = [[J[1, 1], -J[0, 1]], [-J[1, 0], J[0, 0]]]
        else:
            cof = lambda i, j: (J[(j + 1) % 3, (i + 1) % 3] * J[(j + 2) % 3, (i + 2) % 3] -  # noqa: E731
                                J[(j + 1) % 3, (i + 2) % 3] * J[(j + 2) % 3, (i + 1) % 3])
            rows = [[cof(i, j) for j in range(3)] for i in range(3)]
            det = sum(J[0, k] * rows[k][0] for k in range(3))
        return torch.stack([torch.stack([r / det for r in row]) for row in rows]), det

    def _weights(self, skip=None):
        w = 1.0
        for d in range(self.dim):
            s = [1] * self.dim
            if d != skip:
                s[self.dim - 1 - d] = self.m
                w = w * self.dev(self.b.qw).reshape(s)
        return w

    def apply(self, x):
        dim, n, m, b = self.dim, self.n, self.m, self.b
        u = x.reshape((n,) * dim + (m,) * dim)
        y = torch.zeros_like(u)
        # cells
        grad = []
        for e in range(dim):
            v = u
            for d in range(dim):
                v = _along(self.D if d == e else self.V, v, self._axis(d))
            grad.append(v)
        Ji, det = self._inverse(self._jacobian([b.qx] * dim))
        phys = [sum(Ji[e, a] * grad[e] for e in range(dim)) for a in range(dim)]
        w = det.abs() * self._weights()
        for e in range(dim):
            v = w * sum(Ji[e, a] * phys[a] for a in range(dim))
            for d in range(dim):
                v = _along((self.D if d == e else self.V).T, v, self._axis(d))
            y += v
        # faces
        for d in range(dim):
            y += self._faces(u, d)
        return y.reshape(-1)

    def _faces(self, u, d):
        dim, b = self.dim, self.b
        ax_c = self._axis(d, nodes=False)
        side = []
        for f in (0, 1):
            x = [b.qx] * dim
            x[d] = np.array([float(f)])
            tabs = [(self.dev(b.fv[f][None]), self.dev(b.fd[f][None])) if e == d else (self.V, self.D)
                    for e in range(dim)]
            Ji, det = self._inverse(self._jacobian(x))
            # J^{-T} e_d points to increasing x_d; surface element |det J| |J^{-T} e_d|
            nrm = Ji[d] / Ji[d].norm(dim=0)
            dS = det.abs() * Ji[d].norm(dim=0) * self._weights(skip=d)
            first = [slice(None)] * dim + [slice(0, 1)] * dim
            hinv = (Ji[d] * nrm).sum(0).abs()[tuple(first)]
            side.append({"J": Ji, "n": nrm, "dS": dS, "h": hinv, "tabs": tabs})
        tr = []
        for f in (0, 1):
            s = side[f]
            val = u
            for e in range(dim):
                val = _along(s["tabs"][e][0], val, self._axis(e))
            c = (s["J"] * s["n"]).sum(1)  # J^{-1} n
            dn = 0
            for g in range(dim):
                v = u
                for e in range(dim):
                    v = _along(s["tabs"][e][1 if e == g else 0], v, self._axis(e))
                dn = dn + c[g] * v
            s["c"] = c
            tr.append((val, dn))
        out = torch.zeros_like(u)
        for f in (0, 1):
            s, sg = side[f], 2 * f - 1  # outward normal sg * n
            val, dn = tr[f][0], sg * tr[f][1]
            nb = lambda v: torch.roll(v, -sg, ax_c)  # noqa: E731  (the neighbour's other face)
            jump = val - nb(tr[1 - f][0])
            avg = 0.5 * (dn + sg * nb(tr[1 - f][1]))
            sigma = self.ip * self.gamma * 0.5 * (s["h"] + nb(side[1 - f]["h"]))
            edge = [slice(None)] * (2 * dim)
            edge[ax_c] = slice(-1, None) if f else slice(0, 1)
            edge = tuple(edge)
            half = torch.full_like(jump, 0.5)
            jump[edge], avg[edge], half[edge] = val[edge], dn[edge], 1.0
            sigma[edge] = self.ip * 2 * self.gamma * s["h"][edge]
            v0 = s["dS"] * (sigma * jump - avg)
            v1 = -s["dS"] * half * jump
            terms = [(v0, None)] + [(sg * s["c"][g] * v1, g) for g in range(dim)]
            for v, g in terms:
                for e in range(dim):
                    v = _along(s["tabs"][e][1 if e == g else 0].T, v, self._axis(e))
                out += v
        return out


class _Patches:
    """vertex patches (2^dim cells) and their fast-diagonalization inverses"""

    def __init__(self, case, b, vertices, device):
        dim, n, m = case["dim"], case["n"], len(b.nodes)
        self.dim, self.n, self.m = dim, n, m
        self.n_comp = dim if case["mesh"] == "elastic" else 1
        self.device = device
        v = np.stack(np.meshgrid(*[np.arange(1, n)] * dim, indexing="ij")[::-1], -1).reshape(-1, dim)
        self.v = v
        h = self._lengths(b, vertices) if vertices is not None else np.full((len(v), dim, 2), 1.0 / n)
        bound = np.stack([v == 1, v == n - 1], -1)
        rows = np.concatenate([h, bound], -1).reshape(-1, 4)
        uniq, inv = (rows, np.arange(len(rows))) if vertices is not None else \
            np.unique(rows, axis=0, return_inverse=True)
        inv = torch.from_numpy(inv.reshape(-1, dim)).to(device)
        coefs = {False: (MU, 2 * MU), True: (2 * MU + LAMBDA, 2 * MU + LAMBDA)} \
            if self.n_comp > 1 else {False: (1.0, 1.0)}
        self.solvers = []  # [component][direction] -> (S [P, K, K], lam [P, K])
        made = {k: self._eigen(b, uniq, IP[case["mesh"]], *ab) for k, ab in coefs.items()}
        for c in range(self.n_comp):
            self.solvers.append([tuple(x[inv[:, d]] for x in made[self.n_comp > 1 and c == d])
                                 for d in range(dim)])
        # DoF indices [P, K^dim] in the level vector, first direction fastest
        K = 2 * m
        i = np.arange(K)
        idx = 0
        for d in range(dim):
            shape = [-1] + [1] * dim
            shape[dim - d] = K
            dof = (v[:, d, None] - 1 + i // m) * (n ** d * m ** dim) + i % m * m ** d
            idx = idx + torch.from_numpy(dof).to(device).reshape([len(v)] + shape[1:])
        self.idx = idx.reshape(len(v), -1)
        x = v - 1
        s = x & 1
        self.color = torch.from_numpy(2 * (s << np.arange(dim)).sum(1) +
                                      (((x + s) // 2).sum(1) & 1)).to(device)

    def _lengths(self, b, vertices):
        """surrogate lengths: distances of opposite faces, averaged with the
        Gauss-Lobatto rule and over the cells of a slot"""
        dim, n = self.dim, self.n
        X = vertices.reshape((n + 1,) * dim + (dim,))
        out = np.zeros((len(self.v), dim, 2))
        for d in range(dim):
            ax = dim - 1 - d
            E = np.diff(X, axis=ax)  # edges along d: [grid z, y, x][coordinate][points ...]
            for e in range(dim):
                if e != d:
                    lo, hi = (np.take(E, np.arange(n) + k, dim - 1 - e)[..., None] for k in (0, 1))
                    E = lo * (1 - b.nodes) + hi * b.nodes
            cell = np.sqrt((E ** 2).sum(dim))  # lengths at the points of each cell
            for _ in range(dim - 1):
                cell = cell @ b.lobatto_w
            for slot in (0, 1):
                acc = 0
                for corner in range(1 << dim):
                    if (corner >> d) & 1 == slot:
                        at = tuple(self.v[:, e] - 1 + ((corner >> e) & 1) for e in range(dim))
                        acc = acc + cell[at[::-1]]
                out[:, d, slot] = acc / 2 ** (dim - 1)
        return out

    def _eigen(self, b, rows, ip, cons, pen):
        S, lam = [], []
        for at in range(0, len(rows), 1 << 15):
            r = rows[at:at + (1 << 15)]
            M, L = _line_matrices(b, r[:, :2], r[:, 2] > 0, r[:, 3] > 0, ip, cons, pen)
            Ci = np.linalg.inv(np.linalg.cholesky(M))
            CT = np.swapaxes(Ci, -1, -2)
            w, Q = np.linalg.eigh(Ci @ L @ CT)
            S.append(CT @ Q)
            lam.append(w)
        return tuple(torch.from_numpy(np.concatenate(a)).to(self.device) for a in (S, lam))

    def solve(self, r, c, sel):
        """A_j^{-1} r_j for the patches `sel` of component c, r [P', K^dim]"""
        dim, K = self.dim, 2 * self.m
        u = r.reshape((-1,) + (K,) * dim)

        def contract(u, d, transpose):
            S = self.solvers[c][d][0][sel]
            S = S.transpose(1, 2).contiguous() if transpose else S
            w = torch.movedim(u, dim - d, 1)
            shape = w.shape
            w = torch.bmm(S, w.reshape(shape[0], K, -1).contiguous()).reshape(shape)
            return torch.movedim(w, 1, dim - d)

        for d in range(dim):
            u = contract(u, d, True)
        lam = 0
        for d in range(dim):
            shape = [-1] + [1] * dim
            shape[dim - d] = K
            lam = lam + self.solvers[c][d][1][sel].reshape(shape)
        u = u / lam
        for d in range(dim):
            u = contract(u, d, False)
        return u.reshape(len(u), -1)


def exact(case, seed, device="cuda"):
    """run()'s output in 64 bits (None for a solve: its iterate depends on when it stops)"""
    if case["call"] == "solve":
        return None
    vertices = _vertices(case, seed)
    b = _Basis(case["degree"])
    rhs = [v.double() for v in _rhs(case, seed, _dtype(case), device)]
    op = _MovedOperator(case, b, vertices, device) if case["mesh"] == "moved" else \
        _KroneckerOperator(case, b, device)
    if case["call"] == "operator":
        return op.apply(rhs[0])
    if case["call"] == "residual":
        return rhs[0] - op.apply(rhs[1])
    pt = _Patches(case, b, vertices, device)
    x = torch.zeros_like(rhs[0]).reshape(pt.n_comp, -1)
    omega = case["relaxation"]
    if case["call"] == "additive":
        r = rhs[0].reshape(pt.n_comp, -1)
        for c in range(pt.n_comp):
            for sel in torch.arange(len(pt.v), device=device).split(1 << 15):
                u = omega * pt.solve(r[c][pt.idx[sel]], c, sel)
                x[c].index_add_(0, pt.idx[sel].reshape(-1), u.reshape(-1))
        return x.reshape(-1)
    for color in range(2 << case["dim"]):
        sel = torch.nonzero(pt.color == color).reshape(-1)
        if len(sel) == 0:
            continue
        r = rhs[0] if color == 0 else rhs[0] - op.apply(x.reshape(-1))
        r = r.reshape(pt.n_comp, -1)
        for c in range(pt.n_comp):
            x[c][pt.idx[sel]] += omega * pt.solve(r[c][pt.idx[sel]], c, sel)
    return x.reshape(-1)
