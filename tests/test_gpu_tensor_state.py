"""What an apply in the tensor-product form keeps with the operator: buffers under
captured graphs, overlapping precisions, and the potential a replay applies."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from dftfe_amd import fe  # noqa: E402


@pytest.fixture
def small():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dftfe_amd.chfsi import KohnShamOperatorDevice

    prob = fe.build_workload("cube20_p4_n64")
    return prob, KohnShamOperatorDevice(prob)


def _block(prob, B, seed, dtype=torch.float64):
    X = np.random.default_rng(seed).uniform(-1, 1, (prob.M, B))
    X[prob.constrained] = 0.0
    return torch.tensor(X, device="cuda", dtype=dtype)


def _capture(op, X, Y):
    """A graph of Y <- H~ X (Y cleared by a kernel)."""
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        Y.zero_()
        op.HX(X, False, 1.0, Y)
    return graph


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_captured_apply_survives_wider_and_other_applies(small, dtype):
    """A narrow apply is captured after a warm-up; later applies, wider and of the
    other precision, must not move the buffer that its graph writes."""
    prob, op = small
    X = _block(prob, 8, 1, dtype)
    op.apply(_block(prob, 1024, 2, dtype))
    want = op.apply(X)
    Y = torch.zeros_like(X)
    graph = _capture(op, X, Y)
    other = torch.float32 if dtype == torch.float64 else torch.float64
    for B, kind in ((64, dtype), (200, other), (224, dtype)):
        op.apply(_block(prob, B, B, kind))
        fill = torch.full((1 << 24,), 7.0, device="cuda")   # takes what was given back
        Y.fill_(3.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(Y, want), (B, kind)
        del fill


def test_precisions_overlap_on_two_streams(small):
    """FP64 and FP32 applies of one operator use scratch of their own."""
    prob, op = small
    X64, X32 = _block(prob, 64, 3), _block(prob, 64, 4, torch.float32)
    want64, want32 = op.apply(X64), op.apply(X32)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[torch.zeros_like(X) for _ in range(20)] for X in (X64, X32)]
    torch.cuda.synchronize()
    for i in range(20):
        for st, X, Y in zip(streams, (X64, X32), got):
            with torch.cuda.stream(st):
                op.HX(X, False, 1.0, Y[i])
    torch.cuda.synchronize()
    assert all(torch.equal(Y, want64) for Y in got[0])
    assert all(torch.equal(Y, want32) for Y in got[1])
