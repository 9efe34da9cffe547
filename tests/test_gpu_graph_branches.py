"""Graphs of several solves: independent ones on two branches, dependent ones in order."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def noise(seed, *shape):
    g = torch.Generator().manual_seed(seed)
    return torch.view_as_complex(torch.randn(*shape, 2, generator=g, dtype=torch.float64)).cuda()


def plan2d(H, ctx, N, k, prec=None):
    h = 1.0 / (N + 1)
    coef = H.coefficients2d(4, N, N, h, h, np.full(N + 2, k * k, np.complex128))
    if prec is None:
        return H.Plan2D(ctx, N, N, coef)
    plan = H.Plan2D(ctx, N, N, coef, prec)
    plan.set_refine(0.0, 2)
    return plan


def same(a, b):
    return torch.equal(torch.view_as_real(a), torch.view_as_real(b))


def replays(H, ctx, solves, want):
    """Three replays with eager work between them, each against the eager results."""
    graph = H.Graph(ctx, solves)
    for _ in range(3):
        for _, _, out in solves:
            out.fill_(float("nan"))
        graph.launch()
        torch.cuda.synchronize()
        for (_, _, out), w in zip(solves, want):
            assert same(out, w)
        solves[0][0].solve(solves[0][1])   # grows and moves nothing the graph holds
    return graph


# FFT, dense (workspace) and mixed (workspace) plans in every place; one, two
# and more solves; two solves on either side of the size rule
@pytest.mark.parametrize("sizes", [(63,), (63, 100), (300, 511, 63), (100, 127, 130, 63, 33), (511, 515), (512, 200, 40)])
@pytest.mark.parametrize("mixed", [False, True])
def test_independent(sizes, mixed):
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    solves, want = [], []
    for i, N in enumerate(sizes):
        plan = plan2d(H, ctx, N, 3.0 + i, H.PREC_MIXED if mixed and i % 2 == 0 else None)
        F = noise(i, 2, N, N)
        want.append(plan.solve(F).clone())
        solves.append((plan, F, torch.empty_like(F)))
    replays(H, ctx, solves, want)


def test_results_that_feed_later_solves():
    """A chain through the middle of a list, and a result written twice: the caller's order."""
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    a, b = plan2d(H, ctx, 255, 3.0), plan2d(H, ctx, 255, 5.0)
    big = plan2d(H, ctx, 1023, 4.0)
    F, G = noise(1, 4, 255, 255), noise(2, 1, 1023, 1023)
    mid, out = torch.empty_like(F), torch.empty_like(F)
    part = mid[2:]   # an overlap that is not the whole buffer
    first = a.solve(F)
    second = b.solve(first)
    third = a.solve(first[2:].contiguous())
    tail = torch.empty_like(third)
    graph = H.Graph(ctx, [(big, G, torch.empty_like(G)), (a, F, mid), (b, mid, out), (a, part, tail)])
    for _ in range(3):
        mid.fill_(float("nan"))
        out.fill_(float("nan"))
        graph.launch()
        torch.cuda.synchronize()
        assert same(mid, first) and same(out, second) and same(tail, third)
        big.solve(G)


def test_in_place():
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    plans = [plan2d(H, ctx, N, 4.0) for N in (127, 255, 511)]
    F = [noise(i, 3, N, N) for i, N in enumerate((127, 255, 511))]
    want = [p.solve(f).clone() for p, f in zip(plans, F)]
    bufs = [f.clone() for f in F]
    graph = H.Graph(ctx, [(p, b, b) for p, b in zip(plans, bufs)])
    for _ in range(3):
        for b, f in zip(bufs, F):
            b.copy_(f)
        graph.launch()
        torch.cuda.synchronize()
        for b, w in zip(bufs, want):
            assert same(b, w)


def test_no_room_for_two_workspaces():
    """A budget that holds one workspace but not two: one branch, as before."""
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    plans = [plan2d(H, ctx, N, 4.0) for N in (300, 310, 290)]
    F = [noise(i, 2, N, N) for i, N in enumerate((300, 310, 290))]
    want = [p.solve(f).clone() for p, f in zip(plans, F)]
    largest = max(p.workspace_bytes(2) for p in plans)
    H.lib().hh_context_bytes_in_use.restype = ctypes.c_size_t
    used = H.lib().hh_context_bytes_in_use(ctx.h)
    ctx.set_memory_budget(used + largest + largest // 2)
    replays(H, ctx, [(p, f, torch.empty_like(f)) for p, f in zip(plans, F)], want)
