"""Graphs of a few short solves take less than the solves' own graphs."""
import time

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def replay_us(H, ctx, solves):
    graph = H.Graph(ctx, solves)
    times = []
    for _ in range(9):
        torch.cuda.synchronize()
        t = time.perf_counter()
        for _ in range(100):
            graph.launch()
        torch.cuda.synchronize()
        times.append((time.perf_counter() - t) * 1e4)
    graph.close()
    return sorted(times)[4]


# one replay saves the start of all graphs but one, 4 us of about 20 each (0.80
# to 0.85 of the sum); on two branches these lists took 0.92 to 1.13 of it
@pytest.mark.parametrize("sizes", [(63, 63, 63), (40, 63, 100), (127, 127, 127)])
def test_short_lists(sizes):
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    solves = []
    for i, N in enumerate(sizes):
        h = 1.0 / (N + 1)
        coef = H.coefficients2d(4, N, N, h, h, np.full(N + 2, (3.0 + i) ** 2, np.complex128))
        F = torch.ones(1, N, N, dtype=torch.complex128, device="cuda")
        solves.append((H.Plan2D(ctx, N, N, coef), F, torch.empty_like(F)))
    each = sum(replay_us(H, ctx, [s]) for s in solves)
    assert replay_us(H, ctx, solves) <= 0.9 * each
