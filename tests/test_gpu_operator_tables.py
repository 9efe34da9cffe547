"""Operator tables that do not fit the staging memory (8 MiB) at once."""
import os
import subprocess
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# bands alone above 8 MiB (16 x 8191 rows x 96 B); factors of every mode (real
# 7.4 and 17 MB, complex 15; 3D 20 MB); tables below 256 KiB; FP32 forms
@pytest.mark.parametrize("dims,nop,k,threshold,mixed", [
    ((7, 8191), 16, 3.0, None, False), ((7, 8191), 16, 3.0, None, True), ((7, 2047), 60, 3.0 + 1.0j, None, False),
    ((257, 301), 3, 3.0, 0.0, False), ((257, 700), 3, 3.0, 0.0, False), ((257, 301), 3, 3.0 + 1.0j, 0.0, False),
    ((100, 100, 65), 1, 3.0, 0.0, False), ((50, 50, 65), 3, 3.0 + 1.0j, 0.0, False), ((5, 9), 2, 3.0, 0.0, False)])
def test_same_bits_as_alone(dims, nop, k, threshold, mixed):
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    prec = H.PREC_MIXED if mixed else H.PREC_F64
    n, rng = dims[-1], np.random.default_rng(7)

    def operator(o):
        k2 = np.full(n + 2, (k + o) ** 2, np.complex128) * (1 + 0.1 * np.sin(np.arange(n + 2) / n))
        h = [1.0 / (d + 1) for d in dims]
        return H.coefficients2d(4, *dims, *h, k2) if len(dims) == 2 else H.coefficients3d(4, *dims, *h, k2)

    def plan(coefs):
        kind = H.Plan2D if len(dims) == 2 else H.Plan3D
        p = kind(ctx, *dims, coefs, prec)
        if threshold is not None:
            p.set_resonance_threshold(threshold)
        if mixed:
            p.set_refine(0.0, 1)
        return p

    coefs = [operator(o) for o in range(nop)]
    F = torch.from_numpy(rng.standard_normal((nop,) + dims[::-1]) + 1j * rng.standard_normal((nop,) + dims[::-1])).cuda()
    many = plan(coefs)
    for replaced in (False, True):
        if replaced:
            many.set_operators(coefs[::-1])
        got = many.solve(F)
        # more rows than a piece holds: some of the operators, the first and the last among them
        for o in sorted({0, 1 % nop, nop // 2, nop - 1}):
            alone = plan([coefs[nop - 1 - o if replaced else o]])
            want = alone.solve(F[o:o + 1].contiguous())
            assert torch.equal(torch.view_as_real(got[o:o + 1]), torch.view_as_real(want)), o
            r = alone.residual(want, F[o:o + 1].contiguous()).abs().max().item()
            scale = F[o].abs().max().item() + 64 * want.abs().max().item()
            assert r <= 64 * 2.0 ** (-20 if mixed else -53) * n * scale


PEAK = """
import sys
sys.path.insert(0, sys.argv[1])
import numpy as np
from hackathon_amd import helmholtz as H
def kib(what):
    return [int(l.split()[1]) for l in open('/proc/self/status') if l.startswith(what)][0]
ctx, N = H.Context(0), 127
plan = H.Plan3D(ctx, N, N, N, H.coefficients3d(4, N, N, N, 1 / 128, 1 / 128, 1 / 128, np.full(N + 2, 9.0 + 0j)))
size = kib('VmPeak')
plan.set_resonance_threshold(0.0)
print('PEAK', kib('VmPeak') - size)
"""


def test_large_tables_are_not_pinned_whole():
    """Every mode of 127^3 flagged, 62 MiB of factors: the process grows by them,
    by the device's address ranges (two and one times that) and by the staging
    memory, not by 1.5 times the tables."""
    out = subprocess.run([sys.executable, "-c", PEAK, ROOT], stdout=subprocess.PIPE, text=True, timeout=100, check=True)
    grown = int(out.stdout.split("PEAK")[1]) / 1024
    assert grown <= 4 * 127 ** 3 * 32 / 2 ** 20 + 32
