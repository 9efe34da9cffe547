"""Norms of a refinement sweep, gathered by the residual kernels, against the norms of its fields."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def noise(*shape):
    g = torch.Generator().manual_seed(sum(shape))
    return torch.view_as_complex(torch.randn(*shape, 2, generator=g, dtype=torch.float64)).cuda()


def build(H, ctx, dims, batch):
    h = [1.0 / (d + 1) for d in dims]
    k2 = np.full(dims[-1] + 2, 4.0, np.complex128)
    if len(dims) == 2:
        plan = H.Plan2D(ctx, *dims, H.coefficients2d(4, *dims, *h, k2), H.PREC_MIXED)
    else:
        plan = H.Plan3D(ctx, *dims, H.coefficients3d(4, *dims, *h, k2), H.PREC_MIXED)
    return plan, noise(batch, *dims[::-1])


# the smallest grids, one wave and block more or less, ragged tiles in each direction,
# more blocks than slots, both tile widths in 3D
@pytest.mark.parametrize("dims,batch", [((2, 2), 1), ((63, 5), 1), ((255, 9), 2), ((256, 4), 1), ((257, 3), 3),
                                        ((31, 2000), 40), ((2, 2, 2), 1), ((31, 9, 17), 2), ((65, 8, 16), 1),
                                        ((64, 33, 40), 3), ((20, 150, 150), 4)])
def test_relative_residual(dims, batch):
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    plan, F = build(H, ctx, dims, batch)
    for spot in (0, F.numel() // 2, F.numel() - 1):   # the largest value of F at either end and inside
        G = F.clone()
        G.view(-1)[spot] = 50.0 + 20.0j
        for sweeps in (0, 2):
            plan.set_refine(1e-30, sweeps)   # never reached: exactly `sweeps` corrections
            u = plan.solve(G)
            n, rel = plan.last_refine()
            assert n == sweeps
            # the same two maxima from the fields: the residual in FP64 here and stored in FP32 there, one rounding;
            # its own sum of at most 27 products (weights of absolute sum below 16) may be contracted differently
            top = G.abs().max().item()
            r = plan.residual(u, G).abs().max().item() / top
            assert rel == pytest.approx(r, rel=2.0 ** -23, abs=64 * 2.0 ** -53 * (16 * u.abs().max().item() / top + 1))


def test_slots_are_left_zero():
    """A small residual after a large one on the same context: nothing of the first is left."""
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    plan, F = build(H, ctx, (127, 40), 2)
    plan.set_refine(1e-30, 1)
    plan.solve(1e12 * F)
    plan.solve(F)
    first = plan.last_refine()[1]
    plan2, _ = build(H, H.Context(0), (127, 40), 2)
    plan2.set_refine(1e-30, 1)
    plan2.solve(F)
    assert plan2.last_refine()[1] == first
