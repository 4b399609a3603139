"""The work a ChFSI user has this library do, as timed cases with plain 64-bit results.

A case names one kind of call, the mesh it runs on (degree, cells per side, DOF layout) and its
width.  The meshes are the periodic cubes of dftfe_amd/fe.py with the cell sizes and quadrature
rules of the repository's workloads (p = 4: 2.5 bohr, 5 Gauss points; p = 5: 2 bohr, 6 points;
p = 6: 1.875 bohr, 8 points) and their density of atoms.  The geometry of a case is fixed, as it
is within one calculation; wavefunctions, potentials and occupations come from the seed.
"""
import functools
import math

import numpy as np
import torch

from dftfe_amd import chfsi, fe, lib

CELL = {4: 2.5, 5: 2.0, 6: 1.875}    # cell edge (bohr) of each degree's workload
GAUSS = {4: 5, 5: 6, 6: 8}           # Gauss points per direction
DEVICE = "cuda:0"


def listed():
    return [
        # one vector: a Lanczos step, or any matrix-vector use of the operator
        {"name": "hx_vector", "kind": "hx", "p": 4, "n": 8, "cols": 1, "dtype": "fp64", "mode": "unique"},
        # the small workload's filter: 64 states, degree 20, launch latency counts
        {"name": "filter_small", "kind": "filter", "p": 4, "n": 8, "cols": 64, "degree": 20, "mode": "unique"},
        # a ragged block in the layout deal.II numbers (duplicated periodic faces)
        {"name": "hx_ragged_dealii", "kind": "hx", "p": 5, "n": 12, "cols": 250, "dtype": "fp64", "mode": "dealii"},
        # FP64 filter of a mid-sized calculation at the production degree, odd width
        {"name": "filter_mid", "kind": "filter", "p": 6, "n": 10, "cols": 333, "degree": 30, "mode": "unique"},
        # the production apply of the mixed-precision pass: all 1024 columns at once
        {"name": "hx_production_fp32", "kind": "hx", "p": 6, "n": 16, "cols": 1024, "dtype": "fp32", "mode": "unique"},
        # the BF16 apply of the first SCF iterations
        {"name": "hx_bf16", "kind": "hx", "p": 6, "n": 12, "cols": 512, "dtype": "bf16", "mode": "unique"},
        # k-points with uneven band counts filtered together
        {"name": "kpoints_batch", "kind": "kbatch", "p": 4, "n": 8, "cols": 140, "k": 4, "degree": 10, "mode": "unique"},
        # orthonormalisation of a filtered block
        {"name": "orthonormalise", "kind": "cholgs", "p": 5, "n": 12, "cols": 500, "mode": "unique"},
        # electron density from the occupied wavefunctions
        {"name": "density", "kind": "density", "p": 6, "n": 12, "cols": 512, "mode": "unique"},
        # gradient of a filter with respect to the potential and the start vectors
        {"name": "filter_gradient", "kind": "backward", "p": 5, "n": 12, "cols": 256, "degree": 10, "mode": "unique"},
        # cell matrices of a new GGA potential, once per SCF iteration
        {"name": "potential_gga", "kind": "potential", "p": 6, "n": 8, "gga": True, "mode": "unique"},
        # one eigensolve of an SCF iteration and the density that goes on from it
        {"name": "scf_iteration", "kind": "scf", "p": 6, "n": 8, "cols": 192, "degree": 20, "mode": "unique"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["hx", "hx", "hx", "filter", "filter", "kbatch", "cholgs", "density", "backward", "potential", "scf"])
    p = rng.choice([4, 5, 6])
    n = rng.choice({4: [6, 8, 10, 12], 5: [6, 8, 10, 12], 6: [4, 6, 8, 10]}[p])
    c = {"kind": kind, "p": p, "n": n, "mode": rng.choice(["unique", "unique", "dealii"])}
    if kind == "hx":
        c["dtype"] = rng.choice(["fp64", "fp64", "fp32", "fp32", "bf16"])
        c["cols"] = _log(rng, 1, 900)
    elif kind == "filter":
        c["cols"], c["degree"] = _log(rng, 16, 320), rng.randint(8, 30)
    elif kind == "kbatch":
        c |= {"p": 4, "n": rng.choice([6, 8]), "mode": "unique", "cols": _log(rng, 24, 200), "k": rng.randint(2, 5), "degree": rng.randint(6, 12)}
    elif kind == "cholgs":
        c["cols"] = _log(rng, 24, 500)
    elif kind == "density":
        c["cols"] = _log(rng, 16, 500)
    elif kind == "backward":
        c |= {"n": min(n, 8), "cols": _log(rng, 16, 250), "degree": rng.randint(4, 12)}
    elif kind == "potential":
        c |= {"n": min(n, 8), "gga": rng.random() < 0.5}
    else:
        # the smaller spectral radius of lower degrees needs fewer filter steps for the same gain
        c |= {"n": min(n, 8), "cols": _log(rng, 40, 190), "degree": rng.randint(*{4: (6, 10), 5: (8, 14), 6: (12, 20)}[p])}
    return c


@functools.lru_cache(maxsize=3)
def _problem(p, n, mode):
    L = n * CELL[p]
    wl = fe.Workload("case", L, n, p, GAUSS[p], max(1, round(0.004 * L ** 3)), 1, 1, 1, seed=100 * p + n)
    return fe.build_problem(wl, mode)


def _bounds(prob):
    """(a0, bLow, bUp) of a filter: the wanted states lie in [a0, bLow]; bUp bounds the spectrum
    (three times the largest one-dimensional kinetic eigenvalue of a cell, and the projectors)."""
    w = prob.gll_w
    nodes, g = prob.gll_x, prob.gauss_x
    dphi = fe.lagrange_tables(nodes, g)[1]
    k1 = (dphi * prob.wq[:, None]).T @ dphi
    mu = np.linalg.eigvalsh(k1 / np.sqrt(np.outer(w, w)))[-1]
    return -3.0, 1.0, float(math.ceil(1.05 * 1.5 * mu / prob.h ** 2 + 8.0))


def _generator(seed, salt=0):
    return torch.Generator(device=DEVICE).manual_seed(int(seed) * 1009 + salt)


def _block(prob, cols, seed, dtype=torch.float64, salt=0):
    """A start block, uniform in [-1, 1); constrained rows are zero."""
    X = torch.rand(prob.M, cols, generator=_generator(seed, salt), device=DEVICE, dtype=dtype) * 2 - 1
    if len(prob.slave_rows):
        X[torch.as_tensor(prob.slave_rows, device=DEVICE)] = 0
    return X


def _modes(prob, cols, seed):
    """Smooth orthogonal-like wavefunctions (low plane waves with noise): what a solver holds
    after its first passes."""
    g = _generator(seed, 5)
    m = np.array(sorted(np.ndindex(13, 13, 13), key=lambda t: (sum((x - 6) ** 2 for x in t), t))[:max(1, (cols + 1) // 2)]) - 6
    pos = np.zeros((prob.M, 3))
    local = np.stack([prob.gll_x[np.arange(prob.ne) // len(prob.gll_x) ** d % len(prob.gll_x)] for d in range(3)], 1)
    pos[prob.cell_map.ravel()] = ((prob.cell_coords[:, None, :] + local[None]) / prob.wl.n).reshape(-1, 3)
    t = 2 * math.pi * torch.as_tensor(pos, device=DEVICE) @ torch.as_tensor(m.T.astype(float), device=DEVICE)
    X = torch.cat([torch.cos(t), torch.sin(t)], dim=1)[:, :cols].contiguous()
    X += 0.1 * (torch.rand(X.shape, generator=g, device=DEVICE, dtype=X.dtype) - 0.5)
    if len(prob.slave_rows):
        X[torch.as_tensor(prob.slave_rows, device=DEVICE)] = 0
    return X


def _bands(case):
    """Band counts of the k-points: uneven, `cols` on average."""
    c, k = case["cols"], case["k"]
    return [max(1, c + (2 * i - k + 1) * c // (3 * k)) for i in range(k)]


def _kpoints(prob, k):
    rng = np.random.default_rng(77 + k)
    return rng.uniform(-math.pi / prob.wl.L, math.pi / prob.wl.L, size=(k, 3))


def _potential(prob, seed, gga):
    """vJxW (C, nq^3) and, for GGA, gJxW (C, nq^3, 3) of another SCF iteration."""
    rng = np.random.default_rng(seed)
    r = prob.quad_points()
    phase = rng.uniform(0, 2 * math.pi, 3)
    wave = np.cos(2 * math.pi * r / prob.wl.L + phase)
    v = (prob.V_q * (1 + 0.1 * wave.prod(-1)) - 0.3) * prob.jxw_cells
    return v, (0.05 * wave * prob.jxw_cells[..., None] if gga else None)


def prepare(case, seed):
    kind = case["kind"]
    prob = _problem(case["p"], case["n"], case["mode"])
    s = {"kind": kind, "case": case, "prob": prob}
    if kind == "kbatch":
        k = _kpoints(prob, case["k"])
        s["op"] = chfsi.KohnShamOperatorDevice(prob, DEVICE, kpoints=k)
        s["X"] = [_block(prob, b, seed, torch.complex128, i) for i, b in enumerate(_bands(case))]
        a0, lo, up = _bounds(prob)
        s["bounds"] = [(lo, up, a0)] * case["k"]
        return s
    s["op"] = chfsi.KohnShamOperatorDevice(prob, DEVICE)
    if kind == "hx":
        dtype = torch.float64 if case["dtype"] == "fp64" else torch.float32
        s["X"] = _block(prob, case["cols"], seed, dtype)
        s["Y"] = torch.zeros_like(s["X"])
    elif kind in ("filter", "backward"):
        s["X"] = _block(prob, case["cols"], seed)
        s["bounds"] = _bounds(prob)
        if kind == "backward":
            s["Ybar"] = _block(prob, case["cols"], seed, salt=3)
    elif kind in ("cholgs", "density", "scf"):
        s["X"] = _modes(prob, case["cols"], seed)
        s["w"] = _weights(case["cols"])
        if kind == "scf":
            a0, lo, up = _bounds(prob)
            s["solver"] = chfsi.ChebyshevSolverDevice(a0, lo, up, cheby_degree=case["degree"], cheby_block_size=256,
                                                      lanczos_steps=10, lanczos_full_residual_margin=True, filter_precision=lib.FP64)
            s["v0"] = torch.as_tensor(prob.lanczos_start, device=DEVICE)
            s["solver"].set_lanczos_start(s["v0"])
    else:
        s["v"], s["g"] = _potential(prob, seed, case["gga"])
    return s


def _weights(cols):
    """Occupations times spin: filled states, then a smooth Fermi edge."""
    i = torch.arange(cols, dtype=torch.float64, device=DEVICE)
    return 2.0 / (1.0 + torch.exp((i - 0.8 * cols) / (0.03 * cols + 1)))


def run(s):
    kind, op, case = s["kind"], s["op"], s["case"]
    if kind == "hx":
        # dst <- M^{-1/2} dst + H~ src with a cleared dst, as the solver's applies outside the filter
        s["Y"].zero_()
        op.HX(s["X"], False, 1.0, s["Y"], bf16=case["dtype"] == "bf16")
        return s["Y"]
    if kind == "filter":
        a0, lo, up = s["bounds"]
        Y = s["X"].clone()
        chfsi.chebyshev_filter(op, Y, case["degree"], lo, up, a0)
        return Y
    if kind == "kbatch":
        Y = [X.clone() for X in s["X"]]
        chfsi.batch_filter(op, Y, list(range(case["k"])), s["bounds"], case["degree"])
        return Y
    if kind == "cholgs":
        Y = s["X"].clone()
        chfsi.cholgs(op, Y)
        return Y
    if kind == "density":
        return op.density(s["X"], s["w"])
    if kind == "backward":
        a0, lo, up = s["bounds"]
        Xbar, g = op.filter_backward(s["X"], s["Ybar"], case["degree"], lo, up, a0)
        return {"Xbar": Xbar, "V": g}
    if kind == "potential":
        if case["gga"]:
            op.set_potential_gga(s["v"], s["g"])
        else:
            op.set_potential(s["v"])
        return op.cell_matrices()
    # the wavefunctions of a pass are defined up to signs and rotations of close states, so what
    # goes on from them is returned: eigenvalues, residual norms and the density
    X = s["X"].clone()
    s["solver"].reinitSpectrumBounds(*_bounds(s["prob"]))
    ev, res, up = s["solver"].solve(op, X)
    return {"ev": ev, "res": res, "rho": op.density(X, s["w"]), "up": up}


def _apply_flops(prob, cols):
    """Interpolation to the quadrature points and back, and the three kinetic terms, direction
    by direction, of every cell and column; the projectors twice."""
    n, q = len(prob.gll_x), len(prob.gauss_x)
    tensor = 2 * (q * n * n + q * q * n + q ** 3) * n + 7 * n ** 4 + q ** 3
    return 2.0 * cols * (prob.C * tensor + 2 * len(prob.pair_cell) * prob.ne * 4)


def work(case):
    prob = _problem(case["p"], case["n"], case["mode"])
    kind, cols = case["kind"], case.get("cols", 0)
    n, q = len(prob.gll_x), len(prob.gauss_x)
    block = 8.0 * prob.M * cols
    data = 4.0 * prob.C * prob.ne + 8.0 * prob.C * prob.nqc + 8.0 * prob.pair_C.size
    up = 2.0 * prob.C * (q * n * n + q * q * n + q ** 3) * n   # interpolation of one column
    if kind == "hx":
        return {"bytes": 2 * block / (1 if case["dtype"] == "fp64" else 2) + data, "flops": _apply_flops(prob, cols)}
    if kind == "filter":
        return {"bytes": 2 * block + data, "flops": case["degree"] * _apply_flops(prob, cols)}
    if kind == "kbatch":
        total = sum(_bands(case))
        return {"bytes": 32.0 * prob.M * total + data, "flops": 2.0 * case["degree"] * _apply_flops(prob, total)}
    if kind == "cholgs":
        return {"bytes": 2 * block, "flops": 2.0 * prob.M * cols * cols}
    if kind == "density":
        return {"bytes": block + 8.0 * prob.C * prob.nqc, "flops": cols * up}
    if kind == "backward":
        m = case["degree"]
        return {"bytes": 3 * block + data, "flops": 2.0 * m * _apply_flops(prob, cols) + 2.0 * m * cols * up}
    if kind == "potential":
        d = 8.0 * prob.C * prob.nqc * (4 if case["gga"] else 1)
        return {"bytes": d + 8.0 * prob.C * prob.ne ** 2, "flops": 2.0 * prob.C * n ** 6 * (2 if case["gga"] else 1)}
    m = case["degree"]
    return {"bytes": 2 * block + data, "flops": (m + 2) * _apply_flops(prob, cols) + 8.0 * prob.M * cols * cols + cols * up}


# ---- plain 64-bit results ------------------------------------------------------------------


class _Plain:
    """The operator in plain torch: dense cell matrices, gather, batched product, index_add."""

    def __init__(self, prob, k=None):
        dt = torch.float64 if k is None else torch.complex128
        t = lambda a, d=dt: torch.as_tensor(np.ascontiguousarray(a), device=DEVICE).to(d)  # noqa: E731
        self.M, self.C = prob.M, prob.C
        fold = np.arange(prob.M)
        fold[prob.slave_rows] = prob.master_rows
        self.map = t(fold[prob.cell_map], torch.int64)
        self.s = t(prob.inv_sqrt_mass)[:, None]
        N = t(prob.Nq, torch.float64)
        H = 0.5 * t(prob.K_e, torch.float64) + N.T @ (t(prob.vJxW, torch.float64)[:, :, None] * N)
        if k is not None:
            Im = -torch.einsum("d,dij->ij", t(k, torch.float64), t(prob.G_c, torch.float64))
            H = torch.complex(H + 0.5 * float(k @ k) * t(prob.M_c, torch.float64), Im.expand_as(H).contiguous())
        self.H = H.to(dt)
        pa, pc, pC = (prob.pair_atom, prob.pair_cell, prob.pair_C) if k is None else fe.projectors(prob, k)
        self.pc, self.pC, self.nproj = t(pc, torch.int64), t(pC), prob.n_proj
        self.pp = t(4 * np.asarray(pa)[:, None] + np.arange(4), torch.int64).reshape(-1)
        self.V = t(prob.proj_V)[:, None]

    def __call__(self, X):
        Y = torch.zeros_like(X)
        step = max(1, int(2e8) // (self.C * self.map.shape[1]))
        for j in range(0, X.shape[1], step):
            x = self.s * X[:, j:j + step]
            xc = x[self.map]                                           # (C, ne, b)
            yc = torch.matmul(self.H, xc)
            b = x.shape[1]
            if len(self.pc):
                pr = torch.matmul(self.pC.conj().transpose(1, 2).contiguous(), xc[self.pc]).reshape(-1, b)
                w = self.V * torch.zeros(self.nproj, b, dtype=X.dtype, device=DEVICE).index_add_(0, self.pp, pr)
                yc.index_add_(0, self.pc, torch.matmul(self.pC, w[self.pp].reshape(-1, 4, b)))
            y = torch.zeros_like(x).index_add_(0, self.map.reshape(-1), yc.reshape(-1, b))
            Y[:, j:j + step] = self.s * y
        return Y


def _scalars(m, a, b, a0):
    """(alpha1, c, alpha2) of the scaled Chebyshev steps 1..m."""
    e, c = (b - a) / 2, (b + a) / 2
    s1 = e / (a0 - c)
    sigma, out = s1, [(s1 / e, c, 0.0)]
    for _ in range(2, m + 1):
        s2 = 1 / (2 / s1 - sigma)
        out.append((2 * s2 / e, c, -sigma * s2))
        sigma = s2
    return out


def _filter(H, X, m, a, b, a0):
    """All iterates X_0 .. X_m of the filter."""
    it = [X]
    for a1, c, a2 in _scalars(m, a, b, a0):
        Y = a1 * (H(it[-1]) - c * it[-1])
        it.append(Y + a2 * it[-2] if len(it) > 1 else Y)
    return it


def _quad(prob, A, B):
    """sum over columns of A and B interpolated to the quadrature points, per cell."""
    fold = np.arange(prob.M)
    fold[prob.slave_rows] = prob.master_rows
    cm = torch.as_tensor(fold[prob.cell_map], device=DEVICE)
    N = torch.as_tensor(prob.Nq, device=DEVICE)
    out = torch.zeros(prob.C, prob.nqc, dtype=torch.float64, device=DEVICE)
    step = max(1, int(1e8) // (prob.C * prob.nqc))
    for j in range(0, A.shape[1], step):
        a = torch.matmul(N, A[:, j:j + step][cm])
        b = a if A is B else torch.matmul(N, B[:, j:j + step][cm])
        out += (a * b).sum(-1)
    return out


def exact(case, seed):
    kind = case["kind"]
    prob = _problem(case["p"], case["n"], case["mode"])
    if kind == "hx":
        dtype = torch.float64 if case["dtype"] == "fp64" else torch.float32
        return _Plain(prob)(_block(prob, case["cols"], seed, dtype).double())
    if kind == "filter":
        a0, lo, up = _bounds(prob)
        return _filter(_Plain(prob), _block(prob, case["cols"], seed), case["degree"], lo, up, a0)[-1]
    if kind == "kbatch":
        a0, lo, up = _bounds(prob)
        return [_filter(_Plain(prob, k), _block(prob, b, seed, torch.complex128, i), case["degree"], lo, up, a0)[-1]
                for i, (k, b) in enumerate(zip(_kpoints(prob, case["k"]), _bands(case)))]
    if kind == "cholgs":
        X = _modes(prob, case["cols"], seed)
        L = torch.linalg.cholesky(X.T @ X)
        return X @ torch.linalg.inv(L).T
    if kind == "density":
        X = _modes(prob, case["cols"], seed) * torch.sqrt(_weights(case["cols"]))
        return _quad(prob, X, X)
    if kind == "backward":
        a0, lo, up = _bounds(prob)
        m, H = case["degree"], _Plain(prob)
        it = _filter(H, _block(prob, case["cols"], seed), m, lo, up, a0)
        # reverse sweep of x_k = a1 (H x_{k-1} - c x_{k-1}) + a2 x_{k-2}
        bar, nxt = _block(prob, case["cols"], seed, salt=3), torch.zeros_like(it[0])
        g = torch.zeros(prob.C, prob.nqc, dtype=torch.float64, device=DEVICE)
        sc = _scalars(m, lo, up, a0)
        for k in range(m, 0, -1):
            a1, c, a2 = sc[k - 1]
            g += a1 * _quad(prob, H.s * bar, H.s * it[k - 1])
            bar, nxt = a1 * (H(bar) - c * bar) + nxt, a2 * bar
        return {"Xbar": bar, "V": g * torch.as_tensor(prob.jxw_cells, device=DEVICE)}
    if kind == "potential":
        v, g = _potential(prob, seed, case["gga"])
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=DEVICE)  # noqa: E731
        N, H = t(prob.Nq), 0.5 * t(prob.K_e)[None]
        A = t(v)[:, :, None] * N
        if case["gga"]:
            A = A + 2 * torch.einsum("cqd,qid->cqi", t(g), t(prob.Gq))
            H = H + torch.matmul(N.T, A)
            B = torch.einsum("cqd,qid->cqi", t(g), t(prob.Gq))
            return H + 2 * torch.matmul(B.transpose(1, 2).contiguous(), N)
        return H + torch.matmul(N.T, A)
    # one pass: bounds, filter, Cholesky orthonormalisation, Rayleigh-Ritz, residuals, density
    H = _Plain(prob)
    up = _upper(H, torch.as_tensor(prob.lanczos_start, device=DEVICE))
    a0, lo, _ = _bounds(prob)
    X = torch.as_tensor(prob.sqrt_mass, device=DEVICE)[:, None] * _modes(prob, case["cols"], seed)
    X = _filter(H, X, case["degree"], lo, up, a0)[-1]
    X = X @ torch.linalg.inv(torch.linalg.cholesky(X.T @ X)).T
    HX = H(X)
    ev, Q = torch.linalg.eigh(0.5 * (X.T @ HX + HX.T @ X))
    X, HX = X @ Q, HX @ Q
    F = H.s * X * torch.sqrt(_weights(case["cols"]))
    return {"ev": ev, "res": (HX - X * ev).norm(dim=0), "rho": _quad(prob, F, F), "up": up}


def _upper(H, v, steps=10):
    """ceil(theta_max + |f|) of a Lanczos run from v."""
    T = np.zeros((steps, steps))
    v, old, beta = v / v.norm(), torch.zeros_like(v), 0.0
    for j in range(steps):
        f = H(v[:, None])[:, 0] - beta * old
        T[j, j] = float(v @ f)
        f = f - T[j, j] * v
        beta = float(f.norm())
        if j + 1 < steps:
            T[j, j + 1] = T[j + 1, j] = beta
        old, v = v, f / beta
    return float(math.ceil(np.linalg.eigvalsh(T)[-1] + beta))
