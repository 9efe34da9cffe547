"""DST block sizes: every choice of the dispatch computes the same bits."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def both(ctx, run):
    """run() with the automatic block size and with 256-thread blocks."""
    auto = run().clone()
    ctx.set_dst_algorithm(0)
    try:
        return auto, run().clone()
    finally:
        ctx.set_dst_algorithm(-1)


def noise(*shape):
    g = torch.Generator().manual_seed(sum(shape))
    return torch.view_as_complex(torch.randn(*shape, 2, generator=g, dtype=torch.float64)).cuda()


# blocks of 256 threads at the edges of the row rule (192, 193, 319, 320), a
# remainder of lines, one line
@pytest.mark.parametrize("N", [1, 15, 31, 63, 127, 255, 511, 1023])
@pytest.mark.parametrize("blocks", [0, 192, 193, 319, 320])
def test_rows(N, blocks):
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    per = 256 if N < 16 else 4096 // (N + 1)
    x = noise(blocks * per or 1, N)
    for rows in (x, x[:-1] if blocks else x):
        a, b = both(ctx, lambda: ctx.dst_rows(rows))
        assert torch.equal(torch.view_as_real(a), torch.view_as_real(b))


@pytest.mark.parametrize("Nx,Ny,layers", [(1, 15, 3), (31, 31, 127), (31, 31, 128), (63, 63, 127), (70, 63, 64),
                                          (65, 31, 20), (127, 127, 9), (255, 255, 2)])
def test_columns(Nx, Ny, layers):
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    x = noise(layers, Ny, Nx)
    a, b = both(ctx, lambda: ctx.dst2d_layers(x))
    assert torch.equal(torch.view_as_real(a), torch.view_as_real(b))


# planes are dealt to the XCDs eight at a time, the rest in order
@pytest.mark.parametrize("Nx,Ny", [(63, 15), (255, 127), (300, 31)])
@pytest.mark.parametrize("layers", [1, 7, 8, 9, 16, 23])
def test_layers_alone(Nx, Ny, layers):
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    x = noise(layers, Ny, Nx)
    got = ctx.dst2d_layers(x)
    want = torch.stack([ctx.dst2d_layers(x[i:i + 1].contiguous())[0] for i in range(layers)])
    assert torch.equal(torch.view_as_real(got), torch.view_as_real(want))


# FP32 spectra of a mixed-precision solve, around the edges of its row (128 and
# 192 blocks at N + 1 = 256) and wide-tile rules (448 and 1024 blocks at 128)
@pytest.mark.parametrize("dims", [(255, 100, 1), (255, 192 * 16, 1), (255, 193 * 16, 1), (31, 31, 20), (63, 63, 128),
                                  (127, 127, 112), (127, 127, 113), (255, 127, 129), (127, 255, 10)])
def test_single_precision_spectra(dims):
    import numpy as np
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    prec = H.PREC_MIXED
    Nx, Ny, Nz = dims
    if Nz == 1:
        coef = H.coefficients2d(4, Nx, Ny, 1 / (Nx + 1), 1 / (Nx + 1), np.full(Ny + 2, 9.0, np.complex128))
        plan, x = H.Plan2D(ctx, Nx, Ny, coef, prec), noise(1, Ny, Nx)
    else:
        h = 1 / (Nx + 1)
        coef = H.coefficients3d(4, Nx, Ny, Nz, h, h, h, np.full(Nz + 2, 9.0, np.complex128))
        plan, x = H.Plan3D(ctx, Nx, Ny, Nz, coef, prec), noise(1, Nz, Ny, Nx)
    a, b = both(ctx, lambda: plan.solve(x))
    assert torch.equal(torch.view_as_real(a), torch.view_as_real(b))
