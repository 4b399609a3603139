"""The apply and the projection that an operator chooses by itself: a caller can return
to them from a set variant, and the workloads' committed passes hold for them."""
import ctypes as ct
import dataclasses
import json
import os
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from dftfe_amd import fe  # noqa: E402
from dftfe_amd import lib as L  # noqa: E402

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(HERE, "golden"))
from make_golden import fixture_path  # noqa: E402


def _operator(name):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dftfe_amd.chfsi import KohnShamOperatorDevice

    prob = fe.build_workload(name)
    return prob, KohnShamOperatorDevice(prob)


@pytest.mark.parametrize("name", ["cube20_p4_n64", "cube18_p5_n64"])
@pytest.mark.parametrize("prec,dtype", [(L.FP64, torch.float64), (L.FP32, torch.float32)])
def test_variants_can_be_unset(name, prec, dtype):
    prob, op = _operator(name)
    blocks = [torch.tensor(prob.initial_guess(N=B, seed_offset=B), device="cuda", dtype=dtype)
              for B in (1, 24, 512)]
    first = [op.apply(X) for X in blocks]
    op.set_hx_variant(prec, 0)
    op.set_proj_variant(prec, 0)
    assert not all(torch.equal(op.apply(X), Y) for X, Y in zip(blocks, first))
    op.set_hx_variant(prec, -1)
    op.set_proj_variant(prec, -1)
    assert all(torch.equal(op.apply(X), Y) for X, Y in zip(blocks, first))
    with pytest.raises(Exception):
        op.set_hx_variant(prec, -2)
    with pytest.raises(Exception):
        op.set_proj_variant(prec, -2)


@pytest.mark.parametrize("name", ["cube30_p6_n1024", "cube24_p5_n256"])
def test_committed_pass_on_the_default_forms(name):
    """Lanczos bounds and one FP64 pass from the oracle's committed results, with no
    variant set; the same after setting and unsetting one."""
    from dftfe_amd.chfsi import ChebyshevSolverDevice, lanczos_bounds

    prob, op = _operator(name)
    with open(fixture_path(name)) as f:
        gold = json.load(f)
    b = gold["bounds"]
    out = []
    for again in (False, True):
        if again:
            op.set_hx_variant(L.FP64, 0)
            op.set_hx_variant(L.FP64, -1)
        lo, up = lanczos_bounds(op, torch.tensor(prob.lanczos_start, device="cuda"), 10)
        assert (lo, up) == (gold["lanczos"]["lower"], gold["lanczos"]["upper"])
        solver = ChebyshevSolverDevice(b["a0"], b["bLow"], b["bUp"], cheby_block_size=gold["block"],
                                       cheby_degree=gold["degree"], reuse_lanczos_upper=True,
                                       filter_precision=0)
        X = torch.tensor(prob.initial_guess(N=gold["states"]), device="cuda")
        lam, res, _ = solver.solve(op, X)
        assert np.abs(lam - gold["pass1"]["eigenvalues"]).max() <= 1e-10
        assert np.abs(res - gold["pass1"]["residuals"]).max() <= 1e-8
        out.append((X, lam, res))
    assert torch.equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][2], out[1][2])


@pytest.mark.parametrize("name,B", [("cube20_p4_n64", 1024), ("cube18_p5_n64", 64)])
@pytest.mark.parametrize("prec,dtype", [(L.FP64, torch.float64), (L.FP32, torch.float32)])
@pytest.mark.parametrize("gga_first", [False, True])
def test_autotune_keeps_both_forms(name, B, prec, dtype, gga_first):
    """Autotuning (on a block or under a potential that takes the cell matrices, too)
    leaves the tensor form to LDA potentials, and applies through the cell matrices
    run the tile that was the fastest."""
    prob, op = _operator(name)
    g = 0.1 * np.random.default_rng(2).uniform(-1, 1, (prob.C, prob.nqc, 3)) * prob.jxw_cells[..., None]
    X = torch.tensor(prob.initial_guess(N=24, seed_offset=3), device="cuda", dtype=dtype)
    lda = op.apply(X)
    if gga_first:
        op.set_potential_gga(prob.vJxW, g)
    tuned = op.autotune(B)
    op.set_proj_variant(prec, -1)
    op.set_potential(prob.vJxW)
    assert torch.equal(op.apply(X), lda)
    op.set_potential_gga(prob.vJxW, g)
    gga = op.apply(X)
    op.set_hx_variant(prec, tuned["fp64" if prec == L.FP64 else "fp32"])
    assert torch.equal(op.apply(X), gga)
    op.set_hx_variant(prec, 0)
    err = ((op.apply(X) - gga).abs().max() / gga.abs().max()).item()
    assert err < (1e-13 if prec == L.FP64 else 2e-6)
    op.set_hx_variant(prec, -1)
    assert torch.equal(op.apply(X), gga)
    op.set_potential(prob.vJxW)
    assert torch.equal(op.apply(X), lda)


# (columns, precision, cells per side, projectors, whether the dense form is the faster)
LINES = [(512, L.FP32, 8, True, True), (320, L.FP32, 8, True, False), (448, L.FP64, 6, True, False),
         (224, L.FP64, 8, True, True), (192, L.FP64, 8, True, False), (1, L.FP64, 6, False, True),
         (1, L.FP32, 8, False, True), (1, L.FP64, 8, False, False), (1, L.FP64, 6, True, False),
         (2, L.FP64, 6, False, False), (224, L.FP64, 8, False, False)]


@pytest.mark.parametrize("B,prec,n,projectors,dense", LINES)
def test_lines_between_the_forms_at_p4(B, prec, n, projectors, dense):
    """Each side of the lines at which the p = 4 apply leaves the tensor form."""
    from dftfe_amd.chfsi import KohnShamOperatorDevice

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    prob = fe.build_problem(fe.Workload("lines", 2.5 * n, n, 4, 5, 8, 1, 1, 1, seed=60 + n))
    if not projectors:
        prob = dataclasses.replace(prob, pair_atom=prob.pair_atom[:0],
                                   pair_cell=prob.pair_cell[:0], pair_C=prob.pair_C[:0])
    op = KohnShamOperatorDevice(prob)
    dtype = torch.float64 if prec == L.FP64 else torch.float32
    X = torch.tensor(prob.initial_guess(N=B, seed_offset=B), device="cuda", dtype=dtype)
    Y = op.apply(X)
    op.set_hx_variant(prec, 0)
    tile = op.apply(X)
    assert torch.equal(Y, tile) == dense
    assert ((Y - tile).abs().max() / tile.abs().max()).item() < (1e-13 if prec == L.FP64 else 2e-6)


@pytest.mark.parametrize("name,B", [("cube20_p4_n64", 1), ("cube20_p4_n64", 33),
                                    ("cube20_p4_n64", 160), ("cube20_p4_n64", 190),
                                    ("cube18_p5_n64", 70), ("cube18_p6_n64", 1)])
def test_no_allocation_form_in_steps(name, B):
    """chfsi_hx_noalloc runs all cells at once where its scratch holds their sums, in
    steps of columns if need be, with chfsi_hx's bits."""
    prob, op = _operator(name)
    X = torch.tensor(prob.initial_guess(N=B, seed_offset=B), device="cuda")
    D = torch.tensor(prob.initial_guess(N=B, seed_offset=B + 1), device="cuda")
    want, got = D.clone(), D.clone()
    st = ct.c_void_p(torch.cuda.current_stream().cuda_stream)
    for f, Y in ((op.lib.chfsi_hx, want), (op.lib.chfsi_hx_noalloc, got)):
        L.check(f(op.handle, ct.c_void_p(X.data_ptr()), B, ct.c_void_p(Y.data_ptr()), B, B, 0,
                  -0.75, st))
    assert torch.equal(got, want)
