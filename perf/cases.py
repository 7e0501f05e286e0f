"""What the solver is measured on: the calls that a boundary element program
makes through the package's public entry points, over the sizes of the
repository's own configurations (1,280 to 327,680 triangles, depth 3 to 7,
1 to 64 right-hand sides, both precisions of the pass).

Kinds of call:
  matvec    Plan.matvec: one Burton-Miller operator product, what every
            Krylov step of a user's own solver pays.
  matvec_t  Plan.matvec_t: the transposed product of adjoint solvers.
  solve     Plan.rhs_plane_wave + Plan.gmres to 1e-6: one scattering problem.
  sweep     Plan.retune + rhs + warm start + gmres: one step of a frequency
            sweep, which pays the plan's setup as well.
  field     Plan.field: pressure at points off the surface ("tree" through
            the multipole expansions, "direct" by the panel sum).
  adjoint   Plan.adjoint_grad with vertex gradients: one step of a shape or
            impedance optimisation (the forward solution in hand).

Geometry: a geodesic subdivision of the icosahedron (20 nu^2 triangles),
on a sphere or on an ellipsoid with smooth bumps of 5%, whose leaf boxes hold
uneven numbers of elements.  Plans use the package's default parameters.

A product of the FP32 pass holds FP32 numbers widened to complex128; the
cases hand it on as complex64, which loses nothing.
"""
import functools
import math

import numpy as np
import torch

import fmbem_gpu_c_amd as F

C_AIR = 343.0
EPS, SIGMA = 0.05, 1.5       # the plans' default truncation rule
DENSE_MATVEC = 21000         # elements up to which exact() forms the dense product
DENSE_SOLVE = 6000           # and a dense solve


def listed():
    return [
        # the smallest product: a coarse sphere of 1,280 triangles, where launches count
        dict(name="matvec-1k-fp64", kind="matvec", nu=8, shape="sphere", size=0.1, freq=1000.0,
             depth=3, nrhs=1, mixed=False),
        # an ordinary FP64 product at 4 kHz (the differentiation configuration's mesh)
        dict(name="matvec-20k-fp64", kind="matvec", nu=32, shape="sphere", size=0.1, freq=4000.0,
             depth=6, nrhs=1, mixed=False),
        # the FP32 Krylov step of the 5 kHz configuration
        dict(name="matvec-82k-mixed", kind="matvec", nu=64, shape="sphere", size=0.3, freq=5000.0,
             depth=6, nrhs=1, mixed=True),
        # many incident waves at one frequency of the batched workload, uneven boxes
        dict(name="matvec-60k-64rhs-mixed", kind="matvec", nu=55, shape="bumpy", size=0.08,
             freq=8000.0, depth=6, nrhs=64, mixed=True),
        # the benchmark's step: 327,680 triangles, 10 kHz, nine right-hand sides, FP32 pass
        dict(name="matvec-328k-9rhs-mixed", kind="matvec", nu=128, shape="sphere", size=0.5,
             freq=10000.0, depth=7, nrhs=9, mixed=True),
        # the same operator in FP64 with one right-hand side: the residual check of a solve
        dict(name="matvec-328k-fp64", kind="matvec", nu=128, shape="sphere", size=0.5,
             freq=10000.0, depth=7, nrhs=1, mixed=False),
        # the transposed product of an adjoint solve with three right-hand sides
        dict(name="matvec_t-20k-3rhs-mixed", kind="matvec_t", nu=32, shape="sphere", size=0.1,
             freq=4000.0, depth=6, nrhs=3, mixed=True),
        # one small scattering problem from right-hand side to solution
        dict(name="solve-1k-fp64", kind="solve", nu=8, shape="sphere", size=0.1, freq=1000.0,
             depth=3, nrhs=1, mixed=False),
        # one step of a frequency sweep on a mesh of odd size
        dict(name="sweep-10k-fp64", kind="sweep", nu=23, shape="bumpy", size=0.1, freq=2500.0,
             depth=5, nrhs=2, mixed=False),
        # a pressure map: 16,384 points off the 5 kHz sphere
        dict(name="field-tree-82k-16k", kind="field", nu=64, shape="sphere", size=0.3,
             freq=5000.0, depth=6, nrhs=1, points=16384, method="fmm", mixed=False),
        # a few microphones: the direct sum at 32 points
        dict(name="field-direct-82k-32", kind="field", nu=64, shape="sphere", size=0.3,
             freq=5000.0, depth=6, nrhs=1, points=32, method="direct", mixed=False),
        # the gradients of a pressure objective with respect to impedance and shape
        dict(name="adjoint-5k-fp64", kind="adjoint", nu=16, shape="sphere", size=0.1,
             freq=2000.0, depth=4, nrhs=1, points=32, mixed=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec"] * 5 + ["matvec_t", "solve", "sweep", "field", "adjoint"])
    # triangles 1,280 .. 327,680 for products and fields, smaller for the
    # calls that solve
    nu = _log_int(rng, 8, {"solve": 40, "sweep": 32, "adjoint": 20}.get(kind, 128))
    n = 20 * nu * nu
    shape = rng.choice(["sphere", "bumpy"])
    size = rng.uniform(0.08, 0.5)
    # 7.5 to 14 element edges per wavelength
    edge = size * math.sqrt(4 * math.pi / n * 4 / math.sqrt(3))
    freq = round(C_AIR / (edge * rng.uniform(7.5, 14.0)), 1)
    # about 5 to 20 elements in a leaf box
    depth = min(7, max(3, int(round(math.log(n / 20.0, 4) + rng.uniform(-0.3, 0.6)))))
    mixed = kind in ("matvec", "matvec_t") and rng.random() < 0.6
    # right-hand sides: within the work of the largest listed case
    top = {"matvec": 64, "matvec_t": 16, "field": 4}.get(kind, 3)
    top = max(1, min(top, int(1.2e6 / n * (2 if mixed else 1))))
    case = dict(kind=kind, nu=nu, shape=shape, size=round(size, 4), freq=freq, depth=depth,
                nrhs=_log_int(rng, 1, top), mixed=mixed)
    if kind == "field":
        case["method"] = rng.choice(["fmm", "fmm", "direct"])
        most = 16384 if case["method"] == "fmm" else int(min(4096, max(64, 4e7 / n)))
        case["points"] = _log_int(rng, 16, most)
    if kind == "adjoint":
        case["points"] = rng.randint(8, 48)
    return case


# ------------------------------------------------------------------ geometry

@functools.lru_cache(maxsize=4)
def _geodesic(nu):
    """Unit sphere: each face of the icosahedron cut into nu^2 triangles."""
    g = (1 + math.sqrt(5)) / 2
    ico = np.array([[-1, g, 0], [1, g, 0], [-1, -g, 0], [1, -g, 0], [0, -1, g], [0, 1, g],
                    [0, -1, -g], [0, 1, -g], [g, 0, -1], [g, 0, 1], [-g, 0, -1], [-g, 0, 1]])
    faces = np.array([[0, 11, 5], [0, 5, 1], [0, 1, 7], [0, 7, 10], [0, 10, 11], [1, 5, 9],
                      [5, 11, 4], [11, 10, 2], [10, 7, 6], [7, 1, 8], [3, 9, 4], [3, 4, 2],
                      [3, 2, 6], [3, 6, 8], [3, 8, 9], [4, 9, 5], [2, 4, 11], [6, 2, 10],
                      [8, 6, 7], [9, 8, 1]])
    row, col = np.meshgrid(np.arange(nu + 1), np.arange(nu + 1), indexing="ij")
    keep = col <= row
    row, col = row[keep], col[keep]                 # point (row, col) of one face
    at = lambda r, c: r * (r + 1) // 2 + c          # noqa: E731
    r, c = row[row < nu], col[row < nu]
    up = np.stack([at(r, c), at(r + 1, c), at(r + 1, c + 1)], 1)
    r, c = row[(row < nu) & (col < row)], col[(row < nu) & (col < row)]
    down = np.stack([at(r, c), at(r + 1, c + 1), at(r, c + 1)], 1)
    one = np.concatenate([up, down])
    w = np.stack([nu - row, row - col, col], 1)     # whole barycentric weights
    pts = np.einsum("pk,fkx->fpx", w, ico[faces]).reshape(-1, 3)
    tri = (one[None] + (np.arange(20) * len(row))[:, None, None]).reshape(-1, 3)
    # points on shared edges fall together: their whole-weight sums agree to rounding
    key = np.round(pts * 64.0).astype(np.int64)
    key = (key[:, 0] * 1000003 + key[:, 1]) * 1000003 + key[:, 2]
    _, first, back = np.unique(key, return_index=True, return_inverse=True)
    v = pts[first]
    v = v / np.linalg.norm(v, axis=1, keepdims=True)
    tri = back.reshape(-1)[tri]
    a, b, cc = v[tri[:, 0]], v[tri[:, 1]], v[tri[:, 2]]
    inward = np.einsum("ix,ix->i", np.cross(b - a, cc - a), a) < 0
    tri[inward] = tri[inward][:, ::-1]
    return np.ascontiguousarray(v), np.ascontiguousarray(tri.astype(np.int32))


def _surface(case):
    """Vertices and outward triangles of the case's surface."""
    v, tri = _geodesic(case["nu"])
    if case["shape"] == "bumpy":
        rng = np.random.default_rng(7)
        r = np.ones(len(v))
        for q in range(4, 10):
            d = rng.standard_normal(3)
            r += 0.05 * math.sqrt(2.0 / 6) * np.cos(q * (v @ (d / np.linalg.norm(d))) + q)
        v = v * r[:, None] * np.array([1.0, 0.875, 1.25])
    return case["size"] * v, tri


def _wavenumber(case):
    return 2 * math.pi * case["freq"] / C_AIR


def _directions(case, seed):
    d = np.random.default_rng([seed, 1]).standard_normal((case["nrhs"], 3))
    return d / np.linalg.norm(d, axis=1, keepdims=True)


def _points(case, seed):
    """Points in a shell of 1.3 to 3 of the surface's largest radius."""
    rng = np.random.default_rng([seed, 2])
    d = rng.standard_normal((case["points"], 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    r = case["size"] * (1.4 if case["shape"] == "bumpy" else 1.0)
    return d * (r * rng.uniform(1.3, 3.0, case["points"]))[:, None]


def _vectors(case, seed, n):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn((case["nrhs"], n), dtype=torch.complex128, device="cuda", generator=g)


def _surface_pressure(case, seed):
    """Surface pressure of the incident waves in the physical-optics limit:
    twice the wave on the lit side, a tenth of it in the shadow."""
    v, tri = _surface(case)
    t = v[tri]
    n = np.cross(t[:, 0] - t[:, 2], t[:, 1] - t[:, 2])
    d = _directions(case, seed)
    p = np.exp(1j * _wavenumber(case) * (d @ t.mean(1).T))
    return torch.tensor(np.where(d @ n.T < 0, 2.0, 0.1) * p, device="cuda")


def _robin(case, seed, n):
    """Robin coefficients i k Y of a random locally reacting admittance."""
    rng = np.random.default_rng([seed, 3])
    y = rng.uniform(0.05, 0.4, n) + 1j * rng.uniform(-0.2, 0.2, n)
    return torch.tensor(1j * _wavenumber(case) * y, device="cuda")


# -------------------------------------------------------- the measured calls

class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    k = _wavenumber(case)
    v, tri = _surface(case)
    mesh = F.Mesh.from_arrays(v, tri)
    tree = F.Tree(mesh, depth=case["depth"])
    kind, n = case["kind"], tree.n
    prec = F.FMB_MIXED if case["mixed"] else F.FMB_FP64
    robin = _robin(case, seed, n) if kind == "adjoint" else None
    # a sweep's plan holds the previous frequency
    start = k / 1.05 if kind == "sweep" else k
    s.plan = F.Plan(tree, start, robin=robin, precision=prec, nrhs_max=case["nrhs"])
    s.k = k
    if kind in ("matvec", "matvec_t"):
        s.x = _vectors(case, seed, n)
        s.y = torch.empty_like(s.x)
        s.prec = prec
    elif kind == "solve":
        s.dirs = _directions(case, seed)
    elif kind == "sweep":
        s.dirs, s.k0 = _directions(case, seed), start
        s.x0, _ = s.plan.gmres(s.plan.rhs_plane_wave(s.dirs), tol=1e-6)
    elif kind == "field":
        s.dirs, s.pts = _directions(case, seed), _points(case, seed)
        s.x = _surface_pressure(case, seed)
    elif kind == "adjoint":
        s.dirs, s.pts = _directions(case, seed), _points(case, seed)
        s.x, _ = s.plan.gmres(s.plan.rhs_plane_wave(s.dirs), tol=1e-12)
    return s


def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "matvec":
        y = s.plan.matvec(s.x, s.y, prec=s.prec)
        return y.to(torch.complex64) if case["mixed"] else y
    if kind == "matvec_t":
        y = s.plan.matvec_t(s.x, prec=s.prec)
        return y.to(torch.complex64) if case["mixed"] else y
    if kind == "solve":
        b = s.plan.rhs_plane_wave(s.dirs)
        x, _ = s.plan.gmres(b, tol=1e-6)
        return b, x
    if kind == "sweep":
        s.plan.retune(s.k)
        b = s.plan.rhs_plane_wave(s.dirs)
        x0 = s.plan.sweep_guess(s.k0, s.x0, s.dirs)
        x, _ = s.plan.gmres(b, x0=x0, tol=1e-6)
        return b, x
    if kind == "field":
        return s.plan.field(s.x, s.pts, s.dirs, method=case["method"])
    J, g, _, dV, dvn = s.plan.adjoint_grad(s.x, s.pts, s.dirs, tol=1e-12, vertices=True)
    return J, g, dV, dvn


# ------------------------------------------------------------- what it takes

def _order(k, side):
    t0 = EPS * (1.0 - 1.0 / SIGMA) ** 1.5
    lo = 1.0 - math.log(t0) / math.log(SIGMA)
    ka = k * side
    hi = ka + (3.0 * math.log(1.0 / EPS)) ** 1.5 / 2.0 * ka ** (1.0 / 3.0)
    return math.ceil((lo ** 4 + hi ** 4) ** 0.25)


def _pass_work(case):
    """Bytes and flops of one operator product: the near-field rows and the
    two leaf bases read once, the vectors read and written, the rotate-
    coaxial-rotate translations with the rotations split into their even and
    odd halves (32 p^3 / 3 flops each)."""
    n, nrhs, csz = 20 * case["nu"] ** 2, case["nrhs"], 8 if case["mixed"] else 16
    side = 2.0 * case["size"] * (1.3 if case["shape"] == "bumpy" else 1.0)
    k, flops, last, boxes = _wavenumber(case), 0.0, None, 0
    for l in range(2, case["depth"] + 1):
        boxes = min(4.05 * 4 ** l, n)        # boxes that a closed surface meets
        p = _order(k, side * 2.0 ** -l)
        flops += 43.0 * boxes * 32.0 / 3.0 * p ** 3 * nrhs
        if last:
            flops += 2 * boxes * 32.0 / 3.0 * last ** 3 * nrhs
        last = p
    near = 9.0 * n * n / boxes               # elements of the neighbouring boxes
    flops += 8.0 * nrhs * (near + 2.0 * n * last * last)
    return csz * (near + 2.0 * n * last * last) + 32.0 * n * nrhs, flops, near, last


def work(case):
    n, nrhs = 20 * case["nu"] ** 2, case["nrhs"]
    bytes_, flops, near, p = _pass_work(case)
    kind = case["kind"]
    if kind == "solve":                      # about 14 steps to 1e-6
        return {"bytes": 14 * bytes_, "flops": 14 * flops}
    if kind == "sweep":                      # the near field and bases made once as well
        setup = 7 * 60.0 * near + 8 * 60.0 * n * p * p
        return {"bytes": 13 * bytes_, "flops": 12 * flops + setup}
    if kind == "field":
        m = case["points"]
        io = 16.0 * nrhs * (n + m) + 24.0 * m
        if case["method"] == "direct":
            return {"bytes": io + 72.0 * n, "flops": 7.0 * m * n * (50 + 8 * nrhs)}
        # the upward basis, and about 60 boxes of order p at each point
        return {"bytes": io + 16.0 * n * p * p,
                "flops": 8.0 * nrhs * n * p * p + m * 60.0 * p * p * (10 + 8 * nrhs)}
    if kind == "adjoint":                    # about 30 transposed steps, 18 moves of each element
        moves = 18.0 * n * (case["points"] + 2 * near / n) * 7 * 60
        return {"bytes": 30 * bytes_, "flops": 30 * flops + moves}
    return {"bytes": bytes_, "flops": flops}


# --------------------------------------------- the same in plain 64-bit torch

_A1, _B1 = (6 - math.sqrt(15)) / 21, (9 + 2 * math.sqrt(15)) / 21
_A2, _B2 = (6 + math.sqrt(15)) / 21, (9 - 2 * math.sqrt(15)) / 21
_W1, _W2 = (155 - math.sqrt(15)) / 1200, (155 + math.sqrt(15)) / 1200
_FAR = np.array([[1 / 3, 1 / 3, 1 / 3, 9 / 40],
                 [_B1, _A1, _A1, _W1], [_A1, _B1, _A1, _W1], [_A1, _A1, _B1, _W1],
                 [_B2, _A2, _A2, _W2], [_A2, _B2, _A2, _W2], [_A2, _A2, _B2, _W2]])


def _collapsed(order):
    x, w = np.polynomial.legendre.leggauss(order)
    th, rho = np.meshgrid(0.5 + 0.5 * x, 0.5 + 0.5 * x, indexing="ij")
    b0 = rho * (1 - th)
    return np.stack([b0, rho - b0, 1 - rho, 0.5 * np.outer(w, w) * rho], -1).reshape(-1, 4)


class _Panels:
    """The collocation discretisation: element centroids against panel
    integrals of the Helmholtz kernels, in float64 on the GPU."""

    def __init__(self, case):
        self.k = _wavenumber(case)
        v, tri = _surface(case)
        v = torch.tensor(v, device="cuda")
        self.t = v[torch.tensor(tri.astype(np.int64), device="cuda")]       # n x 3 x 3
        a, b, c = self.t[:, 0], self.t[:, 1], self.t[:, 2]
        nn = torch.linalg.cross(a - c, b - c)
        two = torch.linalg.norm(nn, dim=1)
        self.normal, self.area = nn / two[:, None], two / 2
        self.c = self.t.mean(1)
        self.rad = torch.linalg.norm(self.t - self.c[:, None], dim=2).amax(1)
        self.n = len(tri)

    def _terms(self, x, nx, y, ny, collocation):
        """K (and T) integrands at x (with normal nx) from y (normal ny)."""
        d = x - y
        r = torch.sqrt((d * d).sum(-1))
        k, e = self.k, torch.exp(1j * self.k * r) / (4 * math.pi * r)
        rny = -(d * ny).sum(-1) / r
        K = e * (1j * k - 1 / r) * rny
        if not collocation:
            return K
        rnx, dot = (d * nx).sum(-1) / r, (nx * ny).sum(-1)
        T = e / (r * r) * ((3 - (k * r) ** 2 - 3j * k * r) * rnx * rny + (1 - 1j * k * r) * dot)
        return K, T

    def field_rows(self, pts):
        """Rows F[q, j] = integral over panel j of dG/dn_y at point q."""
        out = 0
        for b0, b1, b2, w in _FAR:
            y = b0 * self.t[:, 0] + b1 * self.t[:, 1] + b2 * self.t[:, 2]
            out = out + self._terms(pts[:, None], None, y[None], self.normal[None], False) * w
        return out * self.area[None]

    def rows(self, i0, i1):
        """Rows i0 .. i1 of the rigid Burton-Miller matrix, coupling i / k."""
        alpha = 1j / self.k
        x, nx = self.c[i0:i1], self.normal[i0:i1]
        A = 0
        for b0, b1, b2, w in _FAR:
            y = b0 * self.t[:, 0] + b1 * self.t[:, 1] + b2 * self.t[:, 2]
            K, T = self._terms(x[:, None], nx[:, None], y[None], self.normal[None], True)
            A = A - (K + alpha * T) * w
        A = A * self.area[None]
        gap = torch.cdist(x, self.c, compute_mode="donot_use_mm_for_euclid_dist")
        i, j = torch.nonzero(gap < 2.0 * self.rad[None], as_tuple=True)
        fix = 0
        for b0, b1, b2, w in _collapsed(8):
            y = b0 * self.t[j, 0] + b1 * self.t[j, 1] + b2 * self.t[j, 2]
            K, T = self._terms(x[i], nx[i], y, self.normal[j], True)
            fix = fix - (K + alpha * T) * w
        A[i, j] = fix * self.area[j]
        own = torch.arange(i0, i1, device="cuda")
        A[own - i0, own] = 0.5 - alpha * self._self(i0, i1)
        return A

    def _self(self, i0, i1):
        """Hypersingular self term at the centroid, as a contour integral."""
        t, c, k = self.t[i0:i1], self.c[i0:i1], self.k
        gx, gw = np.polynomial.legendre.leggauss(24)
        osc, inv = 0, 0
        for e in range(3):
            P, Q = t[:, e], t[:, (e + 1) % 3]
            L = torch.linalg.norm(Q - P, dim=1)
            u = (Q - P) / L[:, None]
            tp = ((c - P) * u).sum(1)
            h = torch.linalg.norm(P + tp[:, None] * u - c, dim=1)
            a, b = torch.atan2(-tp, h), torch.atan2(L - tp, h)
            inv = inv + (torch.sin(b) - torch.sin(a)) / h
            for g, w in zip(gx, gw):
                rho = h / torch.cos((a + b) / 2 + (b - a) / 2 * g)
                osc = osc + (b - a) / 2 * w * (torch.exp(1j * k * rho) - 1) / rho
        return -(osc + inv - 2j * math.pi * k) / (4 * math.pi)


def _chunks(n, cols):
    step = max(1, int(3e7 // cols))
    return [(i, min(n, i + step)) for i in range(0, n, step)]


def exact(case, seed):
    kind, n = case["kind"], 20 * case["nu"] ** 2
    if kind in ("matvec", "matvec_t"):
        if n > DENSE_MATVEC:
            return None
        P, x = _Panels(case), _vectors(case, seed, n)
        y = torch.zeros_like(x)
        for i0, i1 in _chunks(n, n):
            A = P.rows(i0, i1)
            if kind == "matvec":
                y[:, i0:i1] = (A @ x.T.contiguous()).T
            else:
                y += x[:, i0:i1] @ A
        return y.to(torch.complex64) if case["mixed"] else y
    if kind in ("solve", "sweep"):
        P, k = _Panels(case), _wavenumber(case)
        d = torch.tensor(_directions(case, seed), device="cuda")
        # e^{ik d.c} + (i/k) d/dn of it
        b = torch.exp(1j * k * (d @ P.c.T)) * (1 - d @ P.normal.T)
        if n > DENSE_SOLVE:
            return b, None
        A = torch.cat([P.rows(i0, i1) for i0, i1 in _chunks(n, n)])
        return b, torch.linalg.solve(A, b.T.contiguous()).T.contiguous()
    if kind == "field":
        if 7.0 * n * case["points"] > 1e10:
            return None
        P, x = _Panels(case), _surface_pressure(case, seed)
        pts = torch.tensor(_points(case, seed), device="cuda")
        d = torch.tensor(_directions(case, seed), device="cuda")
        p = torch.exp(1j * P.k * (d @ pts.T))
        for i0, i1 in _chunks(case["points"], n):
            p[:, i0:i1] += (P.field_rows(pts[i0:i1]) @ x.T.contiguous()).T
        return p
    return None
