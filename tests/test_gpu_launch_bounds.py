"""Batches of more work items than one launch takes: kernels with a grid of tiles hand them to the others, or walk."""

import pytest

from tests._util import flush

pytestmark = pytest.mark.gpu


@pytest.fixture
def room(gpu):
    """About 70 GB of the card's 288 free, given back afterwards."""
    import torch

    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info(gpu)[0] < 100 << 30:
        pytest.skip("needs 100 GB of device memory")
    yield gpu
    torch.cuda.empty_cache()


def _ends(n):
    return [0, 1, n // 2, n - 2, n - 1]


def test_harmonic_table_of_2_30_edges(room):
    flush("harmonic table, 2^30 + 5 edges, l_max 0")
    import torch

    from ye3t_amd.runtime import native

    E = 2 ** 30 + 5
    vec = torch.ones((E, 3), device=room, dtype=torch.float32)
    values, _ = native.real_sph_table(vec, 0, with_gradient=False)
    want, _ = native.real_sph_table(vec[:7].contiguous(), 0, with_gradient=False)
    assert tuple(values.shape) == (E, 1) and torch.equal(values[_ends(E)], want[:5])
    assert bool((values == want[0]).all())


def test_radial_table_of_2_32_edges(room):
    flush("radial table, 2^32 + 131 edges, n_max 0")
    import torch

    from ye3t_amd.runtime import native

    E = 2 ** 32 + 131
    r = torch.full((E,), 2.0, device=room, dtype=torch.float32)
    r[E - 1] = 5.5  # beyond the cutoff
    rc = torch.full((E,), 5.0, device=room, dtype=torch.float32)
    values, _ = native.radial_table(r, rc, rc, 0, with_derivative=False)
    assert values[_ends(E)].flatten().tolist() == [1.0, 1.0, 1.0, 1.0, 0.0]
    assert int(values.sum(dtype=torch.float64)) == E - 1


@pytest.mark.parametrize("form", ["grouped", "shared", "sparse"])
def test_monomials_of_2_29_rows(room, form):
    """x^2 of 2^29 + 7 rows, eight equal outputs and one; the gradient 2 x g."""
    flush(f"{form} monomials, 2^29 + 7 rows")
    import torch

    from ye3t_amd import runtime

    B = 2 ** 29 + 7
    x = torch.full((B, 1), 3.0, device=room, dtype=torch.float32)
    x[B - 1] = 5.0

    def call(v, outputs):
        offs, outs, vals = list(range(outputs + 1)), list(range(outputs)), [1.0] * outputs
        if form == "grouped":
            return runtime.symmetric_power_monomial_contraction(v, [[2]] * outputs, offs, outs, vals)
        if form == "shared":
            return runtime.symmetric_power_shared_monomial_contraction(v, [[2]], offs, [0] * outputs, outs, vals)
        return runtime.symmetric_power_shared_sparse_monomial_contraction(v, [0, 1], [0], [2], offs, [0] * outputs,
                                                                          outs, vals)

    out = call(x, 8)
    assert out[_ends(B)].sum(dim=1).tolist() == [72.0, 72.0, 72.0, 72.0, 200.0]
    assert int(out.sum(dtype=torch.float64)) == 72 * (B - 1) + 200
    del out
    x.requires_grad_(True)
    (g,) = torch.autograd.grad(call(x, 1), x, torch.ones((B, 1), device=room))
    assert g[_ends(B)].flatten().tolist() == [6.0, 6.0, 6.0, 6.0, 10.0]
    assert int(g.sum(dtype=torch.float64)) == 6 * (B - 1) + 10


def test_channels_of_a_schedule_of_140_million(room):
    """More parts of a tile than the second grid axis has."""
    flush("scheduled channels, one edge, 1.4e8 channels")
    import torch

    from ye3t_amd.runtime import native

    K = 140_000_003
    one = lambda *s: torch.full(s, 2.0, device=room, dtype=torch.float32)  # noqa: E731
    zeros = torch.zeros(K, dtype=torch.int64, device=room)
    scales = torch.full((K,), 3.0, device=room)
    scales[K - 1] = 5.0
    values, derivs = native.scheduled_radial_angular_channels(
        one(1, 1), one(1, 1), one(1, 1), one(1, 1, 3), one(1, 3), torch.zeros(1, dtype=torch.int64, device=room),
        zeros, zeros, zeros - 1, scales)
    assert values[0, _ends(K)].tolist() == [12.0, 12.0, 12.0, 12.0, 20.0]
    assert int(values.sum(dtype=torch.float64)) == 12 * (K - 1) + 20
    assert int(derivs.sum(dtype=torch.float64)) == 108 * (K - 1) + 180  # 3 scales of (2 2 2 + 2 2)
