"""Performance cases of the sparse-grid DG operator library.

Each case is one call (or one short run) that a user's program makes through the Python
package: applying an operator, integrating a wave / transport / Vlasov system with RK4,
changing basis, applying an imported sparse matrix, projecting initial data, and
advancing a batch of uneven solves.  `exact` restates every one of them in plain FP64
torch / numpy from the definitions (multiwavelets, central flux, collocation points).
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from __graft_entry__ import load_package

RANGES = {  # what `draw` covers
    "D": (1, 6), "k": (1, 5), "n": (1, 10), "N": (60, 3_000_000), "steps": (1, 200),
    "work": 1.2e8,  # state entries x steps x right-hand-side weight of one drawn run
}


def listed():
    return [
        # the smallest product: an integrator written in Python, one right-hand side a call
        dict(name="apply_transport_2d", do="apply", op="transport", D=2, k=2, n=4, prec="fp64"),
        # the 2-D wave configuration of the benchmark: a small solve of 200 steps
        dict(name="wave_2d_small", do="rk4", op="wave", D=2, k=3, n=5, prec="fp64", steps=200),
        # the 3-D transport configuration, FP32 operator and FP64 state
        dict(name="transport_3d_fp32", do="rk4", op="transport", D=3, k=3, n=7, prec="fp32", steps=100),
        # a large 4-D solve in the FP32 form (2.9 M coefficients)
        dict(name="transport_4d_fp32", do="rk4", op="transport", D=4, k=4, n=8, prec="fp32", steps=10),
        # the largest grid that is served, in plain FP64 (6.8 M coefficients)
        dict(name="transport_4d_fp64", do="rk4", op="transport", D=4, k=4, n=9, prec="fp64", steps=10),
        # a large second-order system in the FP32 form: two operator passes a stage
        dict(name="wave_3d_fp32", do="rk4", op="wave", D=3, k=4, n=9, prec="fp32", steps=20),
        # laplacian_matrix(...) * u at a higher order, an odd number of modes a cell
        dict(name="laplacian_3d_k5", do="apply", op="laplacian", D=3, k=5, n=6, prec="fp64"),
        # the 2 + 2 dimensional Vlasov configuration, free streaming
        dict(name="vlasov_4d", do="vlasov", Dx=2, k=2, n=8, prec="fp32", force=False, steps=10),
        # point values of a solution (output, pointwise products)
        dict(name="modal_to_points_3d", do="transform", frm="modal", to="points", D=3, k=3, n=7),
        # an operator imported as the (m, n, colptr, rowval, nzval) triplet
        dict(name="csc_gradient_3d", do="csc", D=3, k=3, n=6, prec="fp64"),
        # initial data given as a function
        dict(name="project_4d", do="project", D=4, k=3, n=6, broadcast=False),
        # many uneven solves submitted together: set up, advanced, read back
        dict(name="batch_mixed_fp32", do="batch", count=48, nmin=4, nmax=8, prec="fp32", steps=50, pick=1),
    ]


# -- sizes ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _levels(D, n):
    """The sparse grid's multi-levels, dimension 1 fastest."""
    if D == 1:
        return tuple((l,) for l in range(n + 1))
    return tuple(low + (top,) for top in range(n + 1) for low in _levels(D - 1, n - top))


@functools.lru_cache(maxsize=None)
def _cells(D, n):
    """Cells of the sparse grid."""
    one = [1 << max(l - 1, 0) for l in range(n + 1)]
    c = one
    for _ in range(D - 1):
        c = [sum(c[i] * one[s - i] for i in range(s + 1)) for s in range(n + 1)]
    return sum(c)


def _size(D, k, n):
    return _cells(D, n) * k ** D


def _draw_grid(rng, kmin=1, kmax=5, Ds=(1, 2, 3, 4, 5, 6), cap=RANGES["N"][1]):
    lo = math.log(RANGES["N"][0])
    while True:
        D, k = rng.choice(Ds), rng.randint(kmin, kmax)
        want = math.exp(rng.uniform(lo, math.log(cap)))
        n = min(range(1, RANGES["n"][1] + 1), key=lambda m: abs(math.log(_size(D, k, m) / want)))
        if RANGES["N"][0] <= _size(D, k, n) <= cap:
            return D, k, n


def draw(rng):
    do = rng.choice(["apply", "apply", "rk4", "rk4", "rk4", "vlasov", "transform", "csc", "project", "batch"])
    prec = rng.choice(["fp64", "fp32"])
    if do == "apply":
        D, k, n = _draw_grid(rng)
        return dict(do=do, op=rng.choice(["transport", "laplacian", "wave", "deriv"]), D=D, k=k, n=n, prec=prec)
    if do == "rk4":
        D, k, n = _draw_grid(rng)
        op = rng.choice(["transport", "wave"])
        weight = _size(D, k, n) * (1 if op == "transport" else 2 * D)
        most = max(1, min(RANGES["steps"][1], int(RANGES["work"] / weight)))
        return dict(do=do, op=op, D=D, k=k, n=n, prec=prec, steps=rng.randint(max(1, most // 4), most))
    if do == "vlasov":
        Dx = rng.choice([1, 2])
        k = rng.choice([2, 2, 3])
        n = rng.randint(3, 9) if Dx == 1 else rng.randint(2, 8 if k == 2 else 6)
        return dict(do=do, Dx=Dx, k=k, n=n, prec=prec, force=rng.random() < 0.5, steps=rng.randint(2, 10))
    if do == "transform":
        frm, to = rng.choice([("modal", "nodal"), ("nodal", "points"), ("points", "nodal"), ("nodal", "modal"),
                              ("modal", "points"), ("points", "modal")])
        while True:
            D, k, n = _draw_grid(rng, 2, 5, (1, 2, 3, 4), 400_000)
            if k != 4 and n <= 9:
                return dict(do=do, frm=frm, to=to, D=D, k=k, n=n)
    if do == "csc":
        D, k, n = _draw_grid(rng, 1, 4, (1, 2, 3, 4), 60_000)
        return dict(do=do, D=D, k=k, n=n, prec=prec)
    if do == "project":
        D = rng.choice([1, 2, 3, 4])
        k = rng.randint(1, 5)
        cap = 2.0e8 / (2 * (k + 4)) ** D  # cells: the nodes of one projection
        most = max([n for n in range(1, 10) if _cells(D, n) <= cap])
        return dict(do=do, D=D, k=k, n=rng.randint(1, most), broadcast=rng.random() < 0.5)
    nmin = rng.randint(3, 5)
    return dict(do="batch", count=rng.randint(2, 40), nmin=nmin, nmax=rng.randint(nmin, 7), prec=prec,
                steps=rng.randint(5, 50), pick=rng.randint(0, 1 << 20))


# -- 1-D tables (plain numpy) ----------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _wavelets(k):
    """Rows of the k multiwavelets on [-1, 1] over (x^i, sgn(x) x^i), i < k."""
    G = np.zeros((2 * k, 2 * k), dtype=np.longdouble)
    for i in range(2 * k):
        for j in range(2 * k):
            p = i % k + j % k
            if (p % 2 == 0) == ((i < k) == (j < k)):
                G[i, j] = np.longdouble(2) / (p + 1)
    dot = lambda a, b: a @ G @ b
    eye = np.eye(2 * k, dtype=np.longdouble)
    leg = []
    for i in range(k):
        v = eye[i].copy()
        for q in leg:
            v -= dot(eye[i], q) * q
        leg.append(v / np.sqrt(dot(v, v)))
    first = []
    for i in range(k):  # sgn(x) x^i made orthogonal to the polynomials
        v = eye[k + i].copy()
        for q in leg:
            v -= dot(eye[k + i], q) * q
        first.append(v)
    second = [v.copy() for v in first]
    for i in range(k - 1):  # nested moments, subtracting the rows as they came in
        for j in range(i + 1, k):
            second[j] -= dot(second[j], eye[k + i]) / dot(first[i], eye[k + i]) * first[i]
    out = [None] * k
    for i in range(k - 1, -1, -1):
        v = second[i].copy()
        for j in range(i + 1, k):
            v -= dot(second[i], out[j]) * out[j]
        out[i] = v / np.sqrt(dot(v, v))
    return np.array(out, dtype=np.float64)


def _legendre(k, x):
    """The k normalised Legendre polynomials of [0, 1] at x in [0, 1]."""
    t = 2 * x - 1
    p = [np.ones_like(t), t]
    for m in range(1, k):
        p.append(((2 * m + 1) * t * p[m] - m * p[m - 1]) / (m + 1))
    return np.stack([math.sqrt(2 * m + 1) * p[m] for m in range(k)])


def _functions(k, n):
    return [(l, c) for l in range(n + 1) for c in range(1 << max(l - 1, 0))]


def _position_matrix(k, n, values):
    """<position basis i, function j> for hierarchical functions given by
    values(level, t): the k functions of a level at reference coordinates t in [0, 1] of
    their cell.  Row c k + m: Legendre mode m on the c-th of the 2^n finest cells."""
    g, w = np.polynomial.legendre.leggauss(12)
    g, w = (g + 1) / 2, w / 2
    P = _legendre(k, g) * w  # k x 12
    fine = 1 << n
    Q = np.zeros((k * fine, k * fine))
    col = 0
    for l, c in _functions(k, n):
        wide = fine >> max(l - 1, 0)  # finest cells under the function's cell
        t = ((np.arange(wide)[:, None] + g[None, :]) / wide).reshape(-1)
        v = values(l, t).reshape(k, wide, -1)  # modes x cells x points
        blk = np.einsum("mp,jcp->cmj", P, v) * 2.0 ** (-n / 2)
        r0 = c * wide * k
        Q[r0:r0 + wide * k, col:col + k] = blk.reshape(wide * k, k)
        col += k
    return Q


@functools.lru_cache(maxsize=None)
def _hier2pos(k, n):
    rows = _wavelets(k)

    def values(l, t):
        if l == 0:
            return _legendre(k, t)
        x = 2 * t - 1
        pw = np.stack([x ** i for i in range(k)])
        return (rows[:, :k] @ pw + np.sign(x) * (rows[:, k:] @ pw)) * 2.0 ** (l / 2)

    return _position_matrix(k, n, values)


@functools.lru_cache(maxsize=None)
def _derivative_1d(k, n):
    """The periodic central-flux derivative in the hierarchical basis, dense."""
    fine = 1 << n
    g, w = np.polynomial.legendre.leggauss(12)
    g, w = (g + 1) / 2, w / 2
    P = _legendre(k, g)
    left, right = _legendre(k, np.zeros(1))[:, 0], _legendre(k, np.ones(1))[:, 0]
    d = np.zeros_like(P)
    for m in range(k):  # the derivative of a Legendre polynomial is a sum of lower ones
        for j in range(m - 1, -1, -2):
            d[m] += 2 * math.sqrt(2 * m + 1) * math.sqrt(2 * j + 1) * P[j]
    inner = -(d * w) @ P.T  # -<P_i', P_j>
    A = np.zeros((fine, k, fine, k))
    for c in range(fine):
        up, dn = (c + 1) % fine, (c - 1) % fine
        A[c, :, c, :] += inner + 0.5 * np.outer(right, right) - 0.5 * np.outer(left, left)
        A[c, :, up, :] += 0.5 * np.outer(right, left)
        A[c, :, dn, :] -= 0.5 * np.outer(left, right)
    Q = _hier2pos(k, n)
    return Q.T @ (A.reshape(k * fine, k * fine) * fine) @ Q


def _nodal_values(k, l, t):
    """The k hierarchical nodal functions of a level at reference coordinates t of their
    cell (0 outside [0, 1])."""
    inside = (t >= 0) & (t <= 1)
    x = t if l == 0 else 2 * t - 1
    if l == 0:
        if k == 2:
            f = [x, 1 - x]
        else:
            nodes = [j / (k - 1) for j in range(k)]
            f = []
            for i in range(k):
                p = np.ones_like(x)
                for j in range(k):
                    if j != i:
                        p = p * (x - nodes[j]) / (nodes[i] - nodes[j])
                f.append(p)
    elif k == 2:
        f = [np.maximum(0.0, 1 - np.abs(x)), np.where(x < 0, x + 1, 0.0)]
    elif k == 3:
        f = [np.maximum(0.0, -4 * x * (x + 1)), np.maximum(0.0, -4 * x * (x - 1)),
             np.where(x < 0, 2 * (x + 1) * (x + 0.5), 0.0)]
    else:
        b, lo, hi = -128.0 / 3.0, x <= 0, x >= 0
        f = [np.where(lo, b * x * (x + 1) * (x + 0.5) * (x + 0.25), 0.0),
             np.where(lo, b * x * (x + 1) * (x + 0.5) * (x + 0.75), 0.0),
             np.where(hi, b * x * (x - 1) * (x - 0.5) * (x - 0.75), 0.0),
             np.where(hi, b * x * (x - 1) * (x - 0.5) * (x - 0.25), 0.0),
             np.where(x < 0, 32.0 / 3.0 * (x + 1) * (x + 0.75) * (x + 0.5) * (x + 0.25), 0.0)]
    return np.where(inside, np.stack(f), 0.0)


@functools.lru_cache(maxsize=None)
def _transform_1d(k, n, frm, to):
    if (frm, to) in (("points", "nodal"), ("modal", "nodal")):
        return np.linalg.inv(_transform_1d(k, n, to, frm))
    if (frm, to) == ("nodal", "modal"):
        return _hier2pos(k, n).T @ _position_matrix(k, n, lambda l, t: _nodal_values(k, l, t))
    xs = []  # nodal -> points: every function at every collocation point, from its side
    for l in range(n + 1):
        nodes = [j / (k - 1) for j in range(k - 1)] if l == 0 else [(2 * j + 1) / (2 * (k - 1)) for j in range(k - 1)]
        nc = 1 << max(l - 1, 0)
        for c in range(nc):
            xs += [(c + q) / nc + 1e-16 for q in nodes] + [(1.0 if l == 0 else (c + 0.5) / nc) - 1e-16]
    x = np.array(xs)
    cols = [_nodal_values(k, l, x if l == 0 else ((1 << l) * x - (2 * c)) / 2) for l, c in _functions(k, n)]
    return np.concatenate(cols).T.copy()


# -- the D-dimensional grid (plain torch) ------------------------------------------------
class _Grid:
    """Pencils of the sparse grid: for a direction, the columns of 1-D vectors along it,
    grouped by the highest level m they reach (the 1-D operator restricted to the levels
    <= m is its upper left block)."""

    def __init__(self, D, k, n, device):
        self.D, self.k, self.n, self.N, self.device = D, k, n, _size(D, k, n), device
        off, blocks = 0, {}
        for lev in _levels(D, n):
            cells = [1 << max(l - 1, 0) for l in lev]
            size = math.prod(cells) * k ** D
            blocks[lev] = np.arange(off, off + size).reshape(cells[::-1] + [k] * D)
            off += size
        self.pencils = []
        for d in range(D):
            by = {}
            for lev, idx in blocks.items():
                other = lev[:d] + lev[d + 1:]
                rows = np.moveaxis(idx, [D - 1 - d, 2 * D - 1 - d], [0, 1])
                by.setdefault(other, []).append((lev[d], rows.reshape(rows.shape[0] * k, -1)))
            per = {}
            for other, parts in by.items():
                parts.sort(key=lambda p: p[0])
                per.setdefault(n - sum(other), []).append(np.concatenate([p[1] for p in parts]))
            self.pencils.append([(m, torch.as_tensor(np.concatenate(v, axis=1), device=device))
                                 for m, v in sorted(per.items())])

    def along(self, d, M, x):
        """The 1-D matrix M (dense, all levels) along direction d."""
        y = torch.empty_like(x)
        for m, idx in self.pencils[d]:
            r = self.k << m
            y[idx] = M[:r, :r] @ x[idx]
        return y

    def table(self, M):
        return torch.as_tensor(M, device=self.device)

    def transform(self, frm, to, x):
        if sorted((frm, to)) == ["modal", "points"]:
            return self.transform("nodal", to, self.transform(frm, "nodal", x))
        M = self.table(_transform_1d(self.k, self.n, frm, to))
        for d in range(self.D):
            x = self.along(d, M, x)
        return x


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


@functools.lru_cache(maxsize=4)
def _grid(D, k, n):
    return _Grid(D, k, n, _device())


def _rk4(rhs, y, dt, steps):
    for _ in range(steps):
        k1 = rhs(y)
        k2 = rhs(y + dt / 2 * k1)
        k3 = rhs(y + dt / 2 * k2)
        k4 = rhs(y + dt * k3)
        y = y + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
    return y


def _rhs(op, G, a=None):
    A = G.table(_derivative_1d(G.k, G.n))
    if op == "transport":
        return lambda x: -sum(a[d] * G.along(d, A, x) for d in range(G.D))
    if op == "deriv":
        return lambda x: G.along(a, A, x)
    lap = lambda x: sum(G.along(d, A, G.along(d, A, x)) for d in range(G.D))
    if op == "laplacian":
        return lap
    return lambda x: torch.cat([x[G.N:], lap(x[:G.N])])


# -- inputs ------------------------------------------------------------------------------
@functools.lru_cache(maxsize=64)
def _coeffs_1d(k, n, what):
    """1-D hierarchical coefficients of exp(2 pi i m x) (what = m), of a Gaussian around
    1/2 of width what[1], or of exp(2 pi i m x) times that Gaussian."""
    g, w = np.polynomial.legendre.leggauss(24)
    g, w = (g + 1) / 2, w / 2
    fine = 1 << n
    x = (np.arange(fine)[:, None] + g[None, :]) / fine
    m, s = what if isinstance(what, tuple) else (what, None)
    f = np.exp(2j * np.pi * m * x) * (1 if s is None else np.exp(-((x - 0.5) / s) ** 2))
    pos = np.einsum("mp,cp->cm", _legendre(k, g) * w, f).reshape(-1) * 2.0 ** (-n / 2)
    return _hier2pos(k, n).T @ pos


@functools.lru_cache(maxsize=4)
def _index_1d(D, k, n):
    """Per direction, the 1-D index of every coefficient."""
    out = [[] for _ in range(D)]
    for lev in _levels(D, n):
        cells = [1 << max(l - 1, 0) for l in lev]
        for d in range(D):
            base = 0 if lev[d] == 0 else 1 << (lev[d] - 1)
            i = (k * (base + np.arange(cells[d])))[:, None] + np.arange(k)[None, :]
            shape = [1] * (2 * D)
            shape[D - 1 - d], shape[2 * D - 1 - d] = cells[d], k
            out[d].append(np.broadcast_to(i.reshape(shape), cells[::-1] + [k] * D).reshape(-1))
    return [torch.as_tensor(np.concatenate(v), device=_device()) for v in out]


def _separable(D, k, n, terms):
    """The real part of a sum of products of 1-D functions: terms of (amplitude, [what])."""
    idx = _index_1d(D, k, n)
    u = torch.zeros(_size(D, k, n), dtype=torch.float64, device=_device())
    for amp, whats in terms:
        p = torch.as_tensor(complex(amp), dtype=torch.complex128, device=u.device)
        for d in range(D):
            p = p * torch.as_tensor(_coeffs_1d(k, n, whats[d]), device=u.device)[idx[d]]
        u += p.real
    return u


def _fourier(rng, D, k, n, count=4):
    """Seeded Fourier modes, wavenumbers 1..4, amplitudes in (-1, 1), as solutions start."""
    terms = []
    for _ in range(count):
        m = rng.integers(1, 5, D) * rng.choice([-1, 1], D)
        terms.append((rng.uniform(-1, 1) * np.exp(2j * np.pi * rng.uniform()), [int(v) for v in m]))
    return _separable(D, k, n, terms)


def _system(case, seed):
    """Coefficients, time step and initial state of an apply or rk4 case."""
    D, k, n, op = case["D"], case["k"], case["n"], case["op"]
    rng = np.random.default_rng([seed, 1])
    a = [float(v) for v in rng.uniform(-1, 1, D)] if op == "transport" else None
    if op == "deriv":
        a = int(rng.integers(0, D))
    u = _fourier(rng, D, k, n)
    if op == "wave":
        u = torch.cat([u, _fourier(rng, D, k, n)])
    speed = sum(abs(v) for v in a) if op == "transport" else 2.0 * D
    return a, 0.1 * 2.0 ** -n / max(speed, 1e-3), u


def _vlasov(case, seed):
    """Initial distribution (Maxwellian in v, perturbed in x) and the force's point values."""
    Dx, k, n = case["Dx"], case["k"], case["n"]
    D = 2 * Dx
    rng = np.random.default_rng([seed, 2])
    s = float(rng.uniform(0.15, 0.3))
    maxwell = [(0, s)] * Dx
    wave = [int(v) for v in rng.integers(1, 3, Dx)]
    f0 = _separable(D, k, n, [(1.0, [0] * Dx + maxwell), (float(rng.uniform(0.05, 0.2)), wave + maxwell)])
    if not case["force"]:
        return f0, None
    G = _grid(D, k, n)
    F = [G.transform("modal", "points", _separable(D, k, n, [(float(rng.uniform(-1, 1)), wave + [0] * Dx)]))
         for _ in range(Dx)]
    return f0, F


def _gradient_triplet(D, k, n, a):
    """sum_d a_d D_d as a 1-based CSC triplet (host)."""
    A = _derivative_1d(k, n)
    A = np.where(np.abs(A) > 1e-11 * np.abs(A).max(), A, 0.0)
    ri, ci, va = [], [], []
    for d, pencils in enumerate(_Grid(D, k, n, torch.device("cpu")).pencils):
        for m, idx in pencils:
            r = k << m
            i, j = np.nonzero(A[:r, :r])
            idx = idx.numpy()
            ri.append(idx[i].reshape(-1))
            ci.append(idx[j].reshape(-1))
            va.append(np.repeat(a[d] * A[i, j], idx.shape[1]))
    ri, ci, va = np.concatenate(ri), np.concatenate(ci), np.concatenate(va)
    N = _size(D, k, n)
    at, inv = np.unique(ci.astype(np.int64) * N + ri, return_inverse=True)
    va = np.bincount(inv, weights=va)
    colptr = np.concatenate([[0], np.cumsum(np.bincount(at // N, minlength=N))]) + 1
    return N, N, colptr.astype(np.int64), (at % N + 1).astype(np.int64), va


def _csc(case, seed):
    D, k, n = case["D"], case["k"], case["n"]
    rng = np.random.default_rng([seed, 3])
    a = [float(v) for v in rng.uniform(-1, 1, D)]
    return _gradient_triplet(D, k, n, a), _fourier(rng, D, k, n)


def _profile(case, seed):
    """The projected function: a wave packet, as (wavenumbers, phase, width)."""
    rng = np.random.default_rng([seed, 4])
    return [int(v) for v in rng.integers(-2, 3, case["D"])], float(rng.uniform(0, 6)), float(rng.uniform(0.5, 1.0))


def _batch(case, seed):
    """The batch's solves: shapes from the case, data from the seed."""
    shape, rng = np.random.default_rng([case["pick"], 5]), np.random.default_rng([seed, 6])
    out = []
    for _ in range(case["count"]):
        D, k = int(shape.integers(2, 5)), int(shape.integers(2, 5))
        n = int(shape.integers(case["nmin"], case["nmax"] + 1))
        op = "wave" if shape.random() < 0.25 else "transport"
        steps = max(1, int(case["steps"] * shape.uniform(0.5, 1.0)))
        a, dt, u = _system(dict(D=D, k=k, n=n, op=op), int(rng.integers(1 << 30)))
        out.append(dict(op=op, D=D, k=k, n=n, a=a, dt=dt, steps=steps, y0=u))
    return out


# -- the measured calls --------------------------------------------------------------------
def prepare(case, seed):
    g = load_package()
    do, prec = case["do"], case.get("prec")
    if do in ("apply", "rk4"):
        a, dt, u = _system(case, seed)
        D, k, n = case["D"], case["k"], case["n"]
        op = (g.transport_matrix(D, k, n, a, precision=prec) if case["op"] == "transport" else
              g.laplacian_matrix(D, k, n, precision=prec) if case["op"] == "laplacian" else
              g.wave_matrix(D, k, n, precision=prec) if case["op"] == "wave" else
              g.D_matrix(D, a + 1, k, n, precision=prec))
        return dict(do=do, op=op, x=u, dt=dt, steps=case.get("steps"))
    if do == "vlasov":
        f0, F = _vlasov(case, seed)
        op = g.vlasov_operator(case["Dx"], case["k"], case["n"], None if F is None else [f.cpu().numpy() for f in F],
                               precision=prec)
        return dict(do="rk4", op=op, x=f0, dt=0.05 * 2.0 ** -case["n"], steps=case["steps"])
    if do == "transform":
        D, k, n = case["D"], case["k"], case["n"]
        x = _fourier(np.random.default_rng([seed, 7]), D, k, n)
        return dict(do="apply", op=g.transform(D, k, n, case["frm"], case["to"]), x=x)
    if do == "csc":
        A, x = _csc(case, seed)
        return dict(do="apply", op=g.csc_matrix(A, precision=prec), x=x)
    if do == "project":
        m, phase, s = _profile(case, seed)

        def f(X):
            arg = 2 * math.pi * m[0] * X[0] + phase
            r2 = (X[0] - 0.5) ** 2
            for d in range(1, case["D"]):
                arg = arg + 2 * math.pi * m[d] * X[d]
                r2 = r2 + (X[d] - 0.5) ** 2
            return torch.cos(arg) * torch.exp(-r2 / (s * s))

        return dict(do=do, g=g, case=case, f=f)
    solves = _batch(case, seed)
    return dict(do="batch", g=g, prec=prec, solves=[dict(s, y0=s["y0"].cpu().numpy()) for s in solves])


def run(state):
    do = state["do"]
    if do == "apply":
        return state["op"] @ state["x"]
    if do == "rk4":
        y = state["x"].clone()
        return state["op"].rk4(y, state["dt"], state["steps"])
    if do == "project":
        c = state["case"]
        return state["g"].vcoeffs_DG_device(c["D"], c["k"], c["n"], state["f"], device="cuda", broadcast=c["broadcast"])
    b = state["g"].Batch(state["prec"])
    slots = [b.add(s["op"], s["D"], s["k"], s["n"], s["y0"], s["dt"], s["steps"], a=s["a"]) for s in state["solves"]]
    b.run()
    out = [b.get(i) for i in slots]
    b.close()
    return out


# -- what a pass cannot do without -----------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _pairs_1d(k, m, frm, to):
    """Coupled cell pairs of a 1-D operator up to level m."""
    A = _derivative_1d(k, m) if frm == "d" else _transform_1d(k, m, frm, to)
    c = 1 << m
    return int((np.abs(A.reshape(c, k, c, k)).max(axis=(1, 3)) > 1e-9 * np.abs(A).max()).sum())


def _flops(D, k, n, dirs=None, frm="d", to=None):
    """Operations of a 1-D operator along `dirs` directions: 2 k^2 a coupled cell pair and
    fiber."""
    one = [1 << max(l - 1, 0) for l in range(n + 1)]
    c = [1] + [0] * n  # cells of the other directions, by level sum
    for _ in range(D - 1):
        c = [sum(c[i] * one[s - i] for i in range(s + 1)) for s in range(n + 1)]
    pairs = sum(c[s] * _pairs_1d(k, n - s, frm, to) for s in range(n + 1))
    return 2.0 * k * k * k ** (D - 1) * pairs * (D if dirs is None else dirs)


def _work_system(op, D, k, n, steps):
    N = _size(D, k, n)
    if op == "deriv":
        return 16.0 * N, _flops(D, k, n, 1)
    rhs = _flops(D, k, n) * (1 if op == "transport" else 2)
    if op == "wave":
        N *= 2
    if steps is None:
        return 16.0 * N, rhs
    return 16.0 * N * steps, (4 * rhs + 14.0 * N) * steps  # the state read and written once a step


def work(case):
    do = case["do"]
    if do in ("apply", "rk4"):
        b, f = _work_system(case["op"], case["D"], case["k"], case["n"], case.get("steps"))
    elif do == "vlasov":
        D, k, n = 2 * case["Dx"], case["k"], case["n"]
        N, nv = _size(D, k, n), D if case["force"] else case["Dx"]
        there = _flops(D, k, n, frm="modal", to="nodal") + _flops(D, k, n, frm="nodal", to="points")
        back = _flops(D, k, n, frm="points", to="nodal") + _flops(D, k, n, frm="nodal", to="modal")
        f = case["steps"] * 4.0 * (_flops(D, k, n, nv) + nv * there + back + 2 * nv * N)
        b = case["steps"] * 16.0 * N
    elif do == "transform":
        D, k, n = case["D"], case["k"], case["n"]
        legs = [(case["frm"], case["to"])]
        if "nodal" not in legs[0]:
            legs = [(case["frm"], "nodal"), ("nodal", case["to"])]
        b, f = 16.0 * _size(D, k, n), sum(_flops(D, k, n, frm=p, to=q) for p, q in legs)
    elif do == "csc":
        f = _flops(case["D"], case["k"], case["n"])  # the matrix: a value and a column index an entry
        b = f / 2 * 12.0 + 24.0 * _size(case["D"], case["k"], case["n"])
    elif do == "project":
        D, k, n = case["D"], case["k"], case["n"]
        P, cells = 2 * (k + 4), _cells(D, n)
        b = cells * (8.0 * k ** D + 8.0 * P ** D * 2)  # the values at the nodes, written by f and read
        f = cells * sum(2.0 * P ** (d + 1) * k ** (D - d) for d in range(D))
    else:
        b = f = 0.0
        for s in _shapes(case):
            db, df = _work_system(s["op"], s["D"], s["k"], s["n"], s["steps"])
            b, f = b + db, f + df
    return {"bytes": float(b), "flops": float(f)}


def _shapes(case):
    """A batch's solves without their data."""
    shape, out = np.random.default_rng([case["pick"], 5]), []
    for _ in range(case["count"]):
        D, k = int(shape.integers(2, 5)), int(shape.integers(2, 5))
        n = int(shape.integers(case["nmin"], case["nmax"] + 1))
        op = "wave" if shape.random() < 0.25 else "transport"
        out.append(dict(D=D, k=k, n=n, op=op, steps=max(1, int(case["steps"] * shape.uniform(0.5, 1.0)))))
    return out


# -- the same in 64 bits -----------------------------------------------------------------------
def exact(case, seed):
    do = case["do"]
    if do in ("apply", "rk4"):
        a, dt, u = _system(case, seed)
        rhs = _rhs(case["op"], _grid(case["D"], case["k"], case["n"]), a)
        return rhs(u) if do == "apply" else _rk4(rhs, u, dt, case["steps"])
    if do == "vlasov":
        return _exact_vlasov(case, seed)
    if do == "transform":
        x = _fourier(np.random.default_rng([seed, 7]), case["D"], case["k"], case["n"])
        return _grid(case["D"], case["k"], case["n"]).transform(case["frm"], case["to"], x)
    if do == "csc":
        (m, n, colptr, rowval, nzval), x = _csc(case, seed)
        col = torch.as_tensor(np.repeat(np.arange(n), np.diff(colptr)), device=x.device)
        y = torch.zeros(m, dtype=torch.float64, device=x.device)
        return y.index_add_(0, torch.as_tensor(rowval - 1, device=x.device),
                            torch.as_tensor(nzval, device=x.device) * x[col])
    if do == "project":
        m, phase, s = _profile(case, seed)
        return _separable(case["D"], case["k"], case["n"], [(np.exp(1j * phase), [(v, s) for v in m])])
    out = []
    for s in _batch(case, seed):
        rhs = _rhs(s["op"], _grid(s["D"], s["k"], s["n"]), s["a"])
        out.append(_rk4(rhs, s["y0"], s["dt"], s["steps"]).cpu().numpy())
    return out


def _exact_vlasov(case, seed):
    Dx, k, n = case["Dx"], case["k"], case["n"]
    f0, F = _vlasov(case, seed)
    G = _grid(2 * Dx, k, n)
    A = G.table(_derivative_1d(k, n))
    v = []
    for d in range(Dx):  # 2 x - 1 along each velocity direction, from its exact coefficients
        e = torch.zeros_like(f0)
        e[k ** (Dx + d)] = 1 / math.sqrt(3.0)
        v.append(G.transform("modal", "points", e))

    def rhs(f):
        c = -sum(v[d] * G.transform("modal", "points", G.along(d, A, f)) for d in range(Dx))
        if F is not None:
            c = c + sum(F[d] * G.transform("modal", "points", G.along(Dx + d, A, f)) for d in range(Dx))
        return G.transform("points", "modal", c)

    return _rk4(rhs, f0, 0.05 * 2.0 ** -n, case["steps"])
