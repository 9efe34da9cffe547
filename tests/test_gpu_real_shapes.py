"""Real bands on systems of more than 512 rows: the built-in block shapes, against a shape set by hand."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def noise(*shape):
    g = torch.Generator().manual_seed(sum(shape))
    return torch.view_as_complex(torch.randn(*shape, 2, generator=g, dtype=torch.float64)).cuda()


# rows: the ends of the ranges and of a chunk; batches: one, odd and even, and
# either side of the rule by blocks (1023 and 1024 blocks of 8 modes above 768 rows)
@pytest.mark.parametrize("n", [513, 520, 768, 769, 777, 1023, 1024, 1025])
@pytest.mark.parametrize("Nx,batch", [(2, 1), (3, 5), (63, 2), (88, 186), (63, 256)])
@pytest.mark.parametrize("varying", [False, True])
def test_same_bits_for_every_width(n, Nx, batch, varying):
    from hackathon_amd import helmholtz as H
    y = np.arange(n + 2) / (n + 1)
    k2 = (9.0 * (1 + (0.2 * np.sin(2 * np.pi * y) if varying else 0 * y))) ** 2 + 0j
    coef = H.coefficients2d(4, Nx, n, 1 / (Nx + 1), 1 / (n + 1), k2)
    plan = H.Plan2D(H.Context(0), Nx, n, coef)
    x = noise(batch, n, Nx)
    got = plan.solve(x).clone()
    W, P, rows, nr = (ctypes.c_int() for _ in range(4))
    H.lib().hh_plan_get_tri_shape(plan.h, *(ctypes.byref(v) for v in (W, P, rows, nr)))
    assert H.lib().hh_plan_set_tri_shape(plan.h, 1, rows, 1) == H.HH_OK
    want = plan.solve(x)
    assert torch.equal(torch.view_as_real(got), torch.view_as_real(want))
    # the residual of the solution, to the rounding of its own sum and of an elimination of n rows
    r = plan.residual(got, x).abs().max().item()
    scale = x.abs().max().item() + 16 * got.abs().max().item()
    assert r <= 64 * 2.0 ** -53 * n * scale
