"""The scheduled edge channels and their per-centre sums at the edges of their tiles."""

import numpy as np
import pytest

from tests._util import flush

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("edges,NR,NA,K", [(1, 1, 1, 1), (7, 3, 4, 5), (301, 9, 16, 144), (65, 2, 300, 600),
                                           (40, 5, 2000, 70), (33, 3, 4, 1500), (4099, 2, 3, 1)])
def test_channels_equal_the_formula(gpu, dtype, edges, NR, NA, K):
    """Rows and schedule in LDS, rows too long for it, schedules too long for it; every product rounded
    by itself, so equal to Torch's elementwise operations bit for bit."""
    flush(f"scheduled channels {edges} edges, {NR} x {NA} tables, {K} channels, {dtype}")
    import torch

    from ye3t_amd.runtime import native

    real = torch.float64 if dtype == "f64" else torch.float32
    g = torch.Generator().manual_seed(edges)
    rand = lambda *s: torch.randn(s, generator=g, dtype=torch.float64).to(gpu, real)  # noqa: E731
    pick = lambda n, *s: torch.randint(0, n, s, generator=g).to(gpu)  # noqa: E731
    rv, rd, av, ad, u, sc = rand(edges, NR), rand(edges, NR), rand(edges, NA), rand(edges, NA, 3), rand(edges, 3), rand(K)
    types, ri, ai, ct = pick(3, edges), pick(NR, K), pick(NA, K), pick(4, K) - 1
    v, d = native.scheduled_radial_angular_channels(rv, rd, av, ad, u, types, ri, ai, ct, sc)
    r, dr, a, ya = rv[:, ri], rd[:, ri], av[:, ai], ad[:, ai]
    on = ((ct < 0) | (types[:, None] == ct)).to(real)
    assert torch.equal(v, torch.where(on > 0, sc * r * a, torch.zeros_like(r)))
    first = (dr[:, :, None] * u[:, None, :]) * a[:, :, None]
    want = sc[None, :, None] * (first + r[:, :, None] * ya)
    assert torch.equal(d, torch.where(on[:, :, None] > 0, want, torch.zeros_like(want)))


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("atoms,degree,C", [(1, 0, 3), (3, 9, 1), (17, 8, 6), (40, 33, 144), (5, 20, 257)])
def test_sums_and_gather(gpu, dtype, atoms, degree, C):
    """Per-centre sums in edge order and the gather of centre rows, rows of whole and of broken vectors."""
    flush(f"density sums {atoms} atoms, up to {degree} edges, {C} channels, {dtype}")
    import torch

    from ye3t_amd.runtime import density_accumulate, density_accumulate_adjoint

    rng = np.random.default_rng(C)
    real = torch.float64 if dtype == "f64" else torch.float32
    centers = np.repeat(np.arange(atoms), rng.integers(0, degree + 1, atoms))
    values = torch.as_tensor(rng.normal(size=(len(centers), C)), dtype=real)
    want = torch.zeros((atoms, C), dtype=real)
    for e, i in enumerate(centers):  # in order, one rounding a sum
        want[i] += values[e]
    c = torch.as_tensor(centers, device=gpu)
    assert torch.equal(density_accumulate(values.to(gpu), c, atoms).cpu(), want)
    rows = torch.as_tensor(rng.normal(size=(atoms, C)), dtype=real, device=gpu)
    assert torch.equal(density_accumulate_adjoint(rows, c), rows[c])
    shuffled = torch.as_tensor(rng.permutation(len(centers)), device=gpu)
    out = density_accumulate(values.to(gpu)[shuffled], c[shuffled], atoms).cpu()
    assert torch.allclose(out, want, rtol=0, atol=(1e-13 if dtype == "f64" else 1e-5) * max(1, degree))
