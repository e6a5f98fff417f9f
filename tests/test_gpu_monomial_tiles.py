"""The monomial contractions at the edges of their tiles and of what a tile holds, against the oracle."""

import numpy as np
import pytest

import oracle
from tests._util import TOL, column_rel_error, flush

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("rows,D,M,O,C", [
    (1, 1, 1, 1, 1), (63, 3, 6, 5, 17), (65, 5, 70, 9, 315),
    (130, 7, 200, 1, 400),    # one output: one wave forward
    (64, 2, 5, 40, 60),       # many outputs, some of them empty
    (200, 9, 900, 12, 3000),  # a table that is read from memory
    (70, 30, 20, 4, 33),      # few waves a tile
    (66, 130, 12, 3, 20),     # rows too wide for a tile
])
def test_forms_against_the_oracle(gpu, dtype, rows, D, M, O, C):
    """Grouped, shared and sparse forms of one table, rows with one and more zero factors among them."""
    flush(f"monomial tiles {rows} rows, D {D}, {M} monomials, {O} outputs, {C} coefficients, {dtype}")
    import torch

    from ye3t_amd import runtime

    rng = np.random.default_rng(M)
    counts = np.where(rng.random((M, D)) < min(0.6, 4 / D), rng.integers(1, 4, (M, D)), 0)
    offs = np.concatenate([[0], np.sort(rng.integers(0, C + 1, O - 1)), [C]])
    terms, vals = rng.integers(0, M, C), rng.normal(size=C)
    outs = np.repeat(np.arange(O), np.diff(offs))
    # magnitudes near one: the columns are compared by their root mean square
    x = rng.uniform(0.5, 1.5, (rows, D)) * rng.choice([-1, 1], (rows, D))
    x[rows // 2, 0] = 0.0
    x[rows - 1, : min(2, D)] = 0.0
    real = torch.float64 if dtype == "f64" else torch.float32
    xd, gd = torch.as_tensor(x, device=gpu).to(real), torch.as_tensor(rng.normal(size=(rows, O)), device=gpu).to(real)
    xr, gr, vr = xd.double().cpu().numpy(), gd.double().cpu().numpy(), torch.as_tensor(vals).to(real).double().numpy()
    want = oracle.symmetric_power_shared_monomial(xr, counts, offs, terms, vr)
    grad = oracle.symmetric_power_shared_monomial_adjoint(gr, xr, counts, offs, terms, vr)
    support = [np.flatnonzero(c) for c in counts]
    sparse = (np.concatenate([[0], np.cumsum([len(s) for s in support])]), np.concatenate(support),
              np.concatenate([c[s] for c, s in zip(counts, support)]), offs, terms, outs, vals)
    forms = {"monomial": (counts[terms], offs, outs, vals), "shared_monomial": (counts, offs, terms, outs, vals),
             "shared_sparse_monomial": sparse}
    for name, table in forms.items():
        xs = xd.clone().requires_grad_(True)
        out = getattr(runtime, f"symmetric_power_{name}_contraction")(xs, *table)
        (gx,) = torch.autograd.grad(out, xs, gd)
        errs = (column_rel_error(out.detach().cpu().numpy(), want), column_rel_error(gx.cpu().numpy(), grad))
        flush(f"  {name} {errs[0]:.2e} {errs[1]:.2e}")
        assert max(errs) < TOL[dtype]


@pytest.mark.parametrize("rows", [1, 64, 129])
def test_complex_supports_equal_a_real_pair(gpu, rows):
    """Complex sparse tables with real inputs and coefficients give the real kernels' values, and their
    gradient the conjugate rule's: for a factor i the gradient of the real part turns by -i."""
    flush(f"complex monomial tiles, {rows} rows")
    import torch

    from ye3t_amd.runtime.native import SparseMonomialTable

    rng = np.random.default_rng(rows)
    toff, comp, ex = np.array([0, 2, 3, 5]), np.array([0, 2, 1, 1, 2]), np.array([1, 2, 3, 1, 1])
    offs, terms, outs, vals = np.array([0, 2, 4]), np.array([0, 1, 2, 0]), np.array([0, 0, 1, 1]), rng.normal(size=4)
    x = torch.as_tensor(rng.normal(size=(rows, 3)), device=gpu)
    g = torch.as_tensor(rng.normal(size=(rows, 2)), device=gpu)
    real = SparseMonomialTable(3, toff, comp, ex, offs, terms, outs, vals, gpu, torch.float64)
    turned = SparseMonomialTable(3, toff, comp, ex, offs, terms, outs, 1j * vals, gpu, torch.complex128)
    out = turned.forward(x.to(torch.complex128))
    assert torch.allclose(out, 1j * real.forward(x), rtol=1e-14, atol=1e-14)
    grad = turned.adjoint(g.to(torch.complex128), x.to(torch.complex128))
    assert torch.allclose(grad, -1j * real.adjoint(g, x), rtol=1e-13, atol=1e-13)


@pytest.mark.parametrize("dtype,big", [("f32", 1e10), ("f64", 1e75)])
def test_grouped_values_scale_their_monomials(gpu, dtype, big):
    """A value that brings a product into range, which the bare product leaves: forward and gradient start from
    the value."""
    flush(f"grouped monomials in range by their values, {dtype}")
    import torch

    from ye3t_amd import runtime

    real = torch.float64 if dtype == "f64" else torch.float32
    counts, vals = np.array([[3, 2], [0, 3]]), np.array([big ** -2, -(big ** -1)])
    x = torch.tensor([[big, -2 * big]] * 3, dtype=real, device=gpu, requires_grad=True)
    out = runtime.symmetric_power_monomial_contraction(x, counts, np.array([0, 1, 2]), np.array([0, 1]), vals)
    (gx,) = torch.autograd.grad(out, x, torch.ones_like(out))
    want = [12 * big ** 2, -4 * big ** 2 - 12 * big]
    assert torch.allclose(gx.double(), torch.tensor([want] * 3, device=gpu, dtype=torch.float64),
                          rtol=1e-14 if dtype == "f64" else 1e-6, atol=0)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("exponents", [(15, 15), (16, 1), (17, 31), (0, 300)])
def test_exponents_beyond_four_bits(gpu, dtype, exponents):
    """Tables whose exponents are packed into four bits each, and, one too large, tables that are not."""
    flush(f"monomial tiles, exponents {exponents}, {dtype}")
    import torch

    from ye3t_amd import runtime

    rng = np.random.default_rng(sum(exponents))
    counts = np.array([[exponents[0], 0, 2], [0, exponents[1], 1], [1, 1, 0]])
    offs, outs, terms, vals = np.array([0, 2, 4]), np.array([0, 0, 1, 1]), np.array([0, 1, 2, 1]), rng.normal(size=4)
    real = torch.float64 if dtype == "f64" else torch.float32
    x = torch.as_tensor(rng.uniform(0.95, 1.05, (67, 3)) * rng.choice([-1, 1], (67, 3)), device=gpu).to(real)
    g = torch.as_tensor(rng.normal(size=(67, 2)), device=gpu).to(real)
    xr, gr, vr = x.double().cpu().numpy(), g.double().cpu().numpy(), torch.as_tensor(vals).to(real).double().numpy()
    want = oracle.symmetric_power_shared_monomial(xr, counts, offs, terms, vr)
    grad = oracle.symmetric_power_shared_monomial_adjoint(gr, xr, counts, offs, terms, vr)
    for name, table in (("monomial", (counts[terms], offs, outs, vals)), ("shared_monomial", (counts, offs, terms, outs, vals))):
        xs = x.clone().requires_grad_(True)
        out = getattr(runtime, f"symmetric_power_{name}_contraction")(xs, *table)
        (gx,) = torch.autograd.grad(out, xs, g)
        # a power e by squaring carries up to e roundings (each squaring doubles those before it), the other
        # factors and the sum less than eight; a column's largest value is at most sqrt(67) its root mean square
        bound = (max(exponents) + 8) * (2.0 ** -53 if dtype == "f64" else 2.0 ** -24) * 67 ** 0.5
        errs = column_rel_error(out.detach().cpu().numpy(), want), column_rel_error(gx.cpu().numpy(), grad)
        flush(f"  {name} {errs[0]:.2e} {errs[1]:.2e} of {bound:.2e}")
        assert max(errs) < bound
