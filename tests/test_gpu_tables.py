"""The radial and harmonic tables at the edges of their tiles, against the oracle."""

import numpy as np
import pytest

import oracle
from tests._util import column_rel_error, flush
from ye3t_amd.runtime import native

pytestmark = pytest.mark.gpu
# computed in fp64 for both storage types: 1e-12 covers the recurrences, fp32 rounds the result once
TOL = {"f64": 1e-12, "f32": 2e-6}


def _values(rng, edges, dtype, gpu):
    import torch

    real = torch.float64 if dtype == "f64" else torch.float32
    vec = rng.normal(size=(edges, 3)) * rng.uniform(0.5, 2.5, (edges, 1))
    if edges > 2:
        vec[1] = 0.0  # below epsilon
    return torch.as_tensor(vec, dtype=real, device=gpu)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("edges", [1, 31, 33, 64, 65, 257])
def test_harmonic_table_tiles(gpu, dtype, edges):
    flush(f"harmonic table, {edges} edges, {dtype}")
    v = _values(np.random.default_rng(edges), edges, dtype, gpu)
    # 9 runs the general kernel.  The oracle sums the Legendre polynomials' coefficients, whose absolute
    # values add up to about (1 + sqrt 2)^l: times the fp64 rounding 6e-13 at l = 9, 9e-12 at l = 12
    for l_max in range(10):
        y_ref, g_ref = oracle.real_sph_table(v.double().cpu().numpy(), l_max)
        y, g = native.real_sph_table(v, l_max)
        y0, none = native.real_sph_table(v, l_max, with_gradient=False)
        assert none is None and column_rel_error(y0.cpu().numpy(), y.cpu().numpy()) < TOL[dtype]
        assert column_rel_error(y.cpu().numpy(), y_ref) < TOL[dtype], l_max
        # the gradient below epsilon is 1e12 of the others: by itself, and the others without it
        keep = v.norm(dim=1).cpu().numpy() > 0
        g, g_ref = g.cpu().numpy().reshape(edges, -1), np.asarray(g_ref).reshape(edges, -1)
        for part in (keep, ~keep):
            if part.any():
                assert column_rel_error(g[part], g_ref[part]) < TOL[dtype], l_max


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("edges", [1, 127, 128, 129, 700])
def test_radial_table_tiles(gpu, dtype, edges):
    """Every column count, with and without derivatives, radii on both sides of the cutoff, and scalar
    operands filled on the device."""
    flush(f"radial table, {edges} edges, {dtype}")
    import torch

    from ye3t_amd import runtime

    real = torch.float64 if dtype == "f64" else torch.float32
    r = torch.as_tensor(np.random.default_rng(edges).uniform(0.1, 5.5, edges), dtype=real, device=gpu)
    rc, lam = torch.full_like(r, 5.0), torch.full_like(r, 0.5723)
    host = [t.double().cpu().numpy() for t in (r, rc, lam)]
    for n_max in range(16):
        v_ref, d_ref = oracle.radial_table(*host, n_max)
        v, d = runtime.cheb_exp_cos_radial_table_with_derivative(r, 5.0, 0.5723, n_max)
        assert column_rel_error(v.cpu().numpy(), v_ref) < TOL[dtype], n_max
        assert column_rel_error(d.cpu().numpy(), d_ref) < TOL[dtype], n_max
        v0, none = native.radial_table(r, rc, lam, n_max, with_derivative=False)
        assert none is None and torch.equal(v0, v)


@pytest.mark.parametrize("l_max", [0, 3, 6, 8])
def test_harmonic_gradient_of_a_length_that_overflows(gpu, l_max):
    """A vector whose squares overflow: direction zero and gradient zero, as the general kernel (l_max 9) has it."""
    flush(f"harmonic table, |v| beyond the square root of the largest number, l_max {l_max}")
    import torch

    v = torch.tensor([[1e160, -2e160, 3e155], [0.3, -0.4, 0.5], [0.0, 2e170, 0.0]], dtype=torch.float64, device=gpu)
    width = (l_max + 1) ** 2
    y, g = native.real_sph_table(v, l_max)
    y9, g9 = native.real_sph_table(v, 9)
    assert bool((g[[0, 2]] == 0).all()) and bool((g9[[0, 2]] == 0).all())
    assert torch.allclose(y, y9[:, :width], rtol=1e-12, atol=1e-14)
    assert torch.allclose(g[1], g9[1, :width], rtol=1e-12, atol=1e-12)
