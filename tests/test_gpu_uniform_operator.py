"""One band per mode for operators whose table rows are all equal: the same
bits as the form with a band per row, and recorded work follows operators that
are replaced by ones of the other form."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def noise(*shape):
    g = torch.Generator(device="cuda")
    g.manual_seed(sum(shape))
    return torch.complex(*(torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64) for _ in range(2)))


def operator(H, dims, k2):
    h = [1.0 / (n + 1) for n in dims]
    fn = H.coefficients2d if len(dims) == 2 else H.coefficients3d
    return fn(6, *dims, *h, np.full(dims[-1] + 2, k2, np.complex128))


def make(H, ctx, dims, ops, prec):
    return (H.Plan2D if len(dims) == 2 else H.Plan3D)(ctx, *dims, ops, prec)


def per_row(op):
    """The same system in a table whose rows differ: the first row's subdiagonal is never read."""
    op = [v.copy() for v in op]
    op[5 if len(op) == 6 else 11][0] += 1.0
    return op


# rows per thread 4, 8 and 16, one and two right-hand sides per thread, real and complex bands, both precisions
@pytest.mark.parametrize("dims,batch", [((31, 12), 2), ((63, 100), 5), ((127, 1000), 2), ((63, 1500), 3), ((31, 31, 90), 3),
                                        ((31, 15, 200), 1)])
@pytest.mark.parametrize("k2", [150.0, 150.0 + 40.0j])
@pytest.mark.parametrize("mixed", [False, True])
def test_same_bits(dims, batch, k2, mixed):
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    op = operator(H, dims, k2)
    F = noise(batch, *dims[::-1])
    sols = []
    for o in (op, per_row(op)):
        plan = make(H, ctx, dims, o, H.PREC_MIXED if mixed else H.PREC_F64)
        plan.set_refine(0.0, 1)
        sols.append(plan.solve(F))
    assert torch.equal(*sols)


@pytest.mark.parametrize("dims", [(63, 100), (31, 31, 40)])
def test_recorded_solve_follows_the_operator(dims):
    from hackathon_amd import helmholtz as H
    ctx = H.Context(0)
    ops = [operator(H, dims, 150.0)]
    y = np.arange(dims[-1] + 2) / (dims[-1] + 1)
    h = [1.0 / (n + 1) for n in dims]
    fn = H.coefficients2d if len(dims) == 2 else H.coefficients3d
    # every mode through the partitioned kernel in both, so that nothing structural changes
    layered = fn(4, *dims, *h, (0.1 * y).astype(np.complex128))
    ops[0] = fn(4, *dims, *h, np.zeros(dims[-1] + 2, np.complex128))
    F = noise(2, *dims[::-1])
    plan = make(H, ctx, dims, ops, H.PREC_F64)
    out = torch.empty_like(F)
    graph = H.Graph(ctx, [(plan, F, out)])
    for op in (ops[0], layered, ops[0]):
        plan.set_operators([op])
        want = plan.solve(F)
        out.zero_()
        graph.launch()
        assert torch.equal(out, want)
