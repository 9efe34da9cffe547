"""Mode factors computed several modes at a time: the reference's recurrence, mode by mode."""
import numpy as np
import pytest

from hackathon_amd import helmholtz as H


def recurrence2d(rows, lam, n):
    """(L, R, Up) in plain double arithmetic, one mode."""
    out, U, Up = [], 0.0, 0.0
    for q, (bm, am, b, a, bp, ap) in enumerate(rows):
        sub, dia, sup = bm * lam + am, b * lam + a, bp * lam + ap
        L = 0.0 if q == 0 else sub / U
        U = dia if q == 0 else dia - L * Up
        Up = sup
        out.append((L, 1.0 / U, 0.0 if q == n - 1 else sup))
    return out


# one mode, whole groups of four and every remainder
@pytest.mark.parametrize("Nx", [2, 3, 4, 5, 6, 7, 8, 13])
@pytest.mark.parametrize("varying", [False, True])
def test_every_mode(Nx, varying):
    n = 11
    y = np.arange(n + 2)
    k2 = (6.0 * (1 + (0.1 * np.sin(y) if varying else 0 * y))) ** 2 + 0j
    coef = H.coefficients2d(4, Nx, n, 1 / (Nx + 1), 1 / (n + 1), k2)
    bp, ap, b, a, bm, am = (np.asarray(c).real for c in coef)
    lam = 2 * np.cos(np.arange(1, Nx + 1) * np.pi / (Nx + 1))
    for m in range(Nx):
        f, singular = H.operator_mode_factors(2, Nx, n, 1, coef, m)
        want = recurrence2d([tuple(float(c[q]) for c in (bm, am, b, a, bp, ap)) for q in range(n)], float(lam[m]), n)
        assert not singular and not f.imag.any()
        # the eigenvalue may differ by a rounding between the two cosines: a few of the recurrence's own
        assert np.allclose(f.real, want, rtol=1e-13, atol=0)
    modes, singular, kappa = H.operator_modes(2, Nx, n, 1, coef, 0.0)
    assert modes == list(range(Nx)) and not singular and np.isfinite(kappa)
