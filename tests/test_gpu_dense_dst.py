"""Dense DST (N + 1 not a power of two) at the edges of its tiles."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def sine_matrix(N):
    """In extended precision: in FP64 the rounded argument of sin(pi q / (N + 1)) near q = N + 1, where the sine is
    zero, costs more than the bound below allows a whole transform."""
    i = np.arange(1, N + 1)
    pi = np.longdouble("3.14159265358979323846264338327950288")
    return np.sqrt(np.longdouble(2) / (N + 1)) * np.sin(pi * (np.outer(i, i) % (2 * (N + 1))) / (N + 1))


def rounding_bound(absx, N):
    """Elementwise bound of a length-N sum of products: each product takes one rounding of the table, one of
    x_j +- x_{M-j} and at most N of the accumulation; twice that covers the reference's own."""
    return 2 * (N + 4) * 2.0 ** -53 * (absx @ np.abs(sine_matrix(N)))


# odd and even N around the padding of the tables (32 outputs, 64 rows of a
# parity), line counts around 8- and 32-line tiles and past the small-tile rule
@pytest.mark.parametrize("N", [2, 4, 5, 30, 32, 33, 62, 64, 65, 126, 128, 129, 130, 200, 257])
@pytest.mark.parametrize("lines", [1, 7, 9, 33, 4100])
def test_rows(N, lines):
    from hackathon_amd import helmholtz as H
    rng = np.random.default_rng(N * 7919 + lines)
    x = rng.standard_normal((lines, N)) + 1j * rng.standard_normal((lines, N))
    got = H.Context(0).dst_rows(torch.from_numpy(x).cuda()).cpu().numpy()
    S = sine_matrix(N)
    for part in ("real", "imag"):
        v = getattr(x, part)
        assert (np.abs(getattr(got, part) - v @ S) <= rounding_bound(np.abs(v), N)).all()


@pytest.mark.parametrize("Nx,Ny,layers", [(5, 2, 3), (33, 34, 1), (20, 129, 2), (100, 65, 40)])
def test_strided_lines(Nx, Ny, layers):
    from hackathon_amd import helmholtz as H
    rng = np.random.default_rng(Nx * 31 + Ny)
    x = rng.standard_normal((layers, Ny, Nx)) + 1j * rng.standard_normal((layers, Ny, Nx))
    got = H.Context(0).dst2d_layers(torch.from_numpy(x).cuda()).cpu().numpy()
    Sx, Sy = sine_matrix(Nx), sine_matrix(Ny)
    want = np.einsum("kj,ljx->lkx", Sy, x @ Sx)
    # the x pass's bound carried through the y pass, plus the y pass's own
    absx = np.abs(x.real) + np.abs(x.imag)
    first = rounding_bound(absx, Nx)
    second = np.einsum("kj,ljx->lkx", np.abs(Sy), first)
    own = 2 * (Ny + 4) * 2.0 ** -53 * np.einsum("kj,ljx->lkx", np.abs(Sy), absx @ np.abs(Sx))
    assert (np.abs(got - want) <= second + own).all()
