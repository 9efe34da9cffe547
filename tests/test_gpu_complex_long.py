"""Complex bands on long systems: every length that a plan accepts is solved,
on both sides of each width of the block (four modes up to 3408 rows)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# batches: chains beside the elimination (3 x 7) and in a launch of their own (40 x 7, every mode a chain)
@pytest.mark.parametrize("n", [3408, 3409, 4096, 4097, 4100, 6816, 6817, 8191, 8192])
@pytest.mark.parametrize("batch,threshold", [(3, None), (3, 0.0), (40, 0.0)])
def test_residual(n, batch, threshold):
    from hackathon_amd import helmholtz as H
    Nx = 7
    coef = H.coefficients2d(4, Nx, n, 1 / (Nx + 1), 1 / (n + 1), np.full(n + 2, (9 + 0.5j) ** 2))
    plan = H.Plan2D(H.Context(0), Nx, n, coef)
    if threshold is not None:
        plan.set_resonance_threshold(threshold)
        assert plan.mode_info()[0] == Nx
    g = torch.Generator().manual_seed(n)
    x = torch.view_as_complex(torch.randn(batch, n, Nx, 2, generator=g, dtype=torch.float64)).cuda()
    u = plan.solve(x)
    # the residual, to the rounding of its own sum and of an elimination of n rows
    r = plan.residual(u, x).abs().max().item()
    scale = x.abs().max().item() + 16 * u.abs().max().item()
    assert r <= 64 * 2.0 ** -53 * n * scale


def test_3d():
    from hackathon_amd import helmholtz as H
    Nx, Ny, n = 3, 4, 4099
    k2e = np.full(n + 2, (9 + 0.5j) ** 2)
    coef = H.coefficients3d(4, Nx, Ny, n, 1 / (Nx + 1), 1 / (Ny + 1), 1 / (n + 1), k2e)
    plan = H.Plan3D(H.Context(0), Nx, Ny, n, coef)
    g = torch.Generator().manual_seed(n)
    x = torch.view_as_complex(torch.randn(2, n, Ny, Nx, 2, generator=g, dtype=torch.float64)).cuda()
    u = plan.solve(x)
    r = plan.residual(u, x).abs().max().item()
    scale = x.abs().max().item() + 16 * u.abs().max().item()
    assert r <= 64 * 2.0 ** -53 * n * scale
