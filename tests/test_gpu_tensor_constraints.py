"""General affine constraints on uniform cells: the tensor-product apply collects plain
sums on the constrained rows, in the colour launches and with all cells at once.

Every 37th DOF is constrained to two to four others with coefficients of both signs.
Bars as for the graded meshes: FP64 HX 1e-13 relative (max-norm), FP32 2e-6, filter
1e-11, density 1e-12, reverse pass 1e-11."""
import dataclasses

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from dftfe_amd import fe  # noqa: E402
from dftfe_amd import lib as L  # noqa: E402
from oracle import chfsi_oracle as O  # noqa: E402

SHAPES = {4: (4, 5, 10.0), 5: (4, 6, 8.0), 6: (4, 8, 7.5)}   # cells, Gauss points, cube


def _rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.fixture(scope="module", params=list(SHAPES))
def case(request):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dftfe_amd.chfsi import KohnShamOperatorDevice

    p = request.param
    n, nq, L_ = SHAPES[p]
    base = fe.build_problem(fe.Workload("constrained", L_, n, p, nq, 3, 16, 16, 8, seed=70 + p))
    rng = np.random.default_rng(p)
    rows = np.arange(5, base.M, 37)
    free = np.setdiff1d(np.arange(base.M), rows)
    count = rng.integers(2, 5, len(rows))
    ptr = np.concatenate([[0], np.cumsum(count)])
    cols = rng.choice(free, ptr[-1])
    vals = rng.uniform(-0.6, 0.8, ptr[-1])
    constrained = np.zeros(base.M, dtype=bool)
    constrained[rows] = True
    zero = lambda a: np.where(constrained, 0.0, a)  # noqa: E731
    prob = dataclasses.replace(base, constrained=constrained, slave_rows=rows, c_ptr=ptr, c_cols=cols,
                               c_vals=vals, mass=zero(base.mass), sqrt_mass=zero(base.sqrt_mass),
                               inv_sqrt_mass=zero(base.inv_sqrt_mass))
    return prob, O.OracleOperator(prob), KohnShamOperatorDevice(prob)


@pytest.mark.parametrize("B", [1, 5, 24, 2048])
@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-13), (torch.float32, 2e-6)])
def test_apply(case, B, dtype, tol):
    """2048 columns: more than 448 workgroups a colour, so colour launches."""
    prob, ref, op = case
    cols = slice(0, B) if B < 2048 else slice(0, B, 97)
    X = prob.initial_guess(N=B, seed_offset=B)
    Xd = torch.tensor(X, device="cuda", dtype=dtype)
    D = torch.tensor(prob.initial_guess(N=B, seed_offset=B + 1), device="cuda", dtype=dtype)
    want = (prob.inv_sqrt_mass[:, None] * D[:, cols].double().cpu().numpy()
            + 0.5 * ref.apply(Xd[:, cols].double().cpu().numpy()))
    op.HX(Xd, False, 0.5, D)
    assert _rel(D[:, cols].double().cpu().numpy(), want) < tol
    assert not D[torch.tensor(prob.constrained)].any()
    assert not Xd[torch.tensor(prob.constrained)].any()


@pytest.mark.parametrize("N", [8, 96])
def test_filter_and_reverse_pass(case, N):
    from dftfe_amd.chfsi import chebyshev_filter

    prob, ref, op = case
    X = prob.sqrt_mass[:, None] * prob.initial_guess(N=N, seed_offset=N)
    _, up, _, _ = O.lanczos_bounds(ref, prob.lanczos_start, 10)
    args = (5, 1.0, up + 10.0, -3.0)
    want = O.chebyshev_filter(ref.HX, X.copy(), *args)
    for prec, tol in ((L.FP64, 1e-11), (L.FP32, 2e-4)):
        Y = torch.tensor(X, device="cuda")
        chebyshev_filter(op, Y, *args, prec)
        assert _rel(Y.cpu().numpy(), want) < tol
    Ybar = prob.initial_guess(N=N, seed_offset=N + 9)
    got, g = op.filter_backward(torch.tensor(X, device="cuda"), torch.tensor(Ybar, device="cuda"), *args)
    xbar, gw = O.filter_backward(ref, X, Ybar, *args)
    ok = ~prob.constrained
    assert _rel(got.cpu().numpy()[ok], xbar[ok]) < 1e-11
    assert _rel(g.cpu().numpy(), gw) < 1e-11


def test_density(case):
    prob, ref, op = case
    X = prob.initial_guess(N=20, seed_offset=2)
    w = np.random.default_rng(1).uniform(0, 2, 20)
    rho = op.density(torch.tensor(X, device="cuda"), torch.tensor(w))
    assert _rel(rho.cpu().numpy(), O.density_at_quadrature(prob, X, w, spin_factor=1.0)) < 1e-12
