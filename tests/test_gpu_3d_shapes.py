"""Real bands in 3D: the built-in block shapes of the mode solves, against a shape set by hand."""
import ctypes

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def noise(*shape):
    g = torch.Generator().manual_seed(sum(shape))
    return torch.view_as_complex(torch.randn(*shape, 2, generator=g, dtype=torch.float64)).cuda()


# layers: the ends of the ranges and of a chunk; grids on either side of the
# rules by modes (1024) and by blocks of 16 modes (1024)
@pytest.mark.parametrize("n", [64, 65, 81, 128, 129, 145])
@pytest.mark.parametrize("Nx,Ny,batch", [(3, 2, 1), (31, 31, 2), (63, 64, 1), (64, 64, 1), (128, 127, 2), (128, 128, 3)])
def test_same_bits_for_every_width(n, Nx, Ny, batch):
    from hackathon_amd import helmholtz as H
    h = 1.0 / 65
    coef = H.coefficients3d(4, Nx, Ny, n, h, h, h, np.full(n + 2, 9.0, np.complex128))
    plan = H.Plan3D(H.Context(0), Nx, Ny, n, coef)
    x = noise(batch, n, Ny, Nx)
    got = plan.solve(x).clone()
    W, P, rows, nr = (ctypes.c_int() for _ in range(4))
    H.lib().hh_plan_get_tri_shape(plan.h, *(ctypes.byref(v) for v in (W, P, rows, nr)))
    assert H.lib().hh_plan_set_tri_shape(plan.h, 1, rows, 1) == H.HH_OK
    want = plan.solve(x)
    assert torch.equal(torch.view_as_real(got), torch.view_as_real(want))
