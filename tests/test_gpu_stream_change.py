"""A solve on another stream than the one on which the operators were replaced."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def setup(H):
    # 5 MB of factors (every mode a chain): 0.1 ms over the link for the kernel that lays them out
    ctx, Nx, n = H.Context(0), 127, 1200
    ops = [H.coefficients2d(4, Nx, n, 1 / (Nx + 1), 1 / (n + 1), np.full(n + 2, k * k, np.complex128)) for k in (3.0, 5.0)]
    plans = [H.Plan2D(ctx, Nx, n, op) for op in ops]
    for p in plans:
        p.set_resonance_threshold(0.0)
    g = torch.Generator().manual_seed(1)
    F = torch.view_as_complex(torch.randn(1, n, Nx, 2, generator=g, dtype=torch.float64)).cuda()
    want = [p.solve(F).clone() for p in plans]
    torch.cuda.synchronize()
    return ctx, plans[0], ops, F, want


def same(a, b):
    return torch.equal(torch.view_as_real(a), torch.view_as_real(b))


@pytest.mark.parametrize("first,second", [("side", "other"), ("side", "default"), ("default", "side")])
def test_solve_after_replacement(first, second):
    from hackathon_amd import helmholtz as H
    ctx, plan, ops, F, want = setup(H)
    streams = {"default": torch.cuda.default_stream(), "side": torch.cuda.Stream(), "other": torch.cuda.Stream()}
    out = torch.empty_like(F)
    for rep in range(6):
        which = (rep + 1) % 2
        with torch.cuda.stream(streams[first]):
            plan.set_operators(ops[which])
        with torch.cuda.stream(streams[second]):
            plan.solve(F, out=out)
        torch.cuda.synchronize()
        assert same(out, want[which]), rep


def test_recording_after_replacement():
    from hackathon_amd import helmholtz as H
    ctx, plan, ops, F, want = setup(H)
    out, side = torch.empty_like(F), torch.cuda.Stream()
    with torch.cuda.stream(side):
        plan.set_operators(ops[1])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        plan.solve(F, out=out)
    for rep in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert same(out, want[1]), rep
        other = plan.solve(F)
        assert same(other, want[1])
