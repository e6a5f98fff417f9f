"""The device check of index inputs against the same conditions in Torch."""

import pytest

from tests._util import flush

pytestmark = pytest.mark.gpu


def _expect(v, first, limit, ordered):
    if not v.numel():
        return (0, 0, False, False)
    return (int(v[0]), int(v[-1]), bool(((v < first) | (v >= limit)).any()),
            bool(ordered and (v[1:] < v[:-1]).any()))


@pytest.mark.parametrize("atoms,edges", [(1, 1), (5, 0), (3, 255), (300, 257), (2049, 70001), (70001, 513)])
def test_check_indices_finds_each_fault_at_every_end(gpu, atoms, edges):
    """No fault in clean input; each kind of fault at the first, middle and last place is found, and only that kind."""
    flush(f"index checks, {atoms} atoms, {edges} edges")
    import torch

    from ye3t_amd.runtime import native, validate_density_csr

    g = torch.Generator().manual_seed(atoms)
    cuts = torch.sort(torch.randint(0, edges + 1, (atoms - 1,), generator=g)).values
    offsets = torch.cat([torch.zeros(1, dtype=torch.int64), cuts, torch.tensor([edges])]).to(gpu)
    nbr = torch.randint(0, atoms, (edges,), generator=g).to(gpu)
    species = torch.randint(0, 4, (atoms,), generator=g).to(gpu, torch.int32)

    def look(o, n, s):
        checks = ((o, native.INT64_MIN, native.INT64_MAX, True), (n, 0, atoms, False), (s, 0, 4, False))
        got = native.check_indices(*checks)
        assert got == [_expect(t.cpu(), *rest) for t, *rest in checks]
        return [got[0][3], got[1][2], got[2][2]]

    assert look(offsets, nbr, species) == [False, False, False]
    assert validate_density_csr(offsets, nbr, atoms, edges, species=species, species_count=4)
    for at in {0, edges // 2, edges - 1} if edges else ():
        for value in (-1, atoms, 2 ** 40):
            bad = nbr.clone()
            bad[at] = value
            assert look(offsets, bad, species)[1]
            with pytest.raises(ValueError, match="neighbor index"):
                validate_density_csr(offsets, bad, atoms, edges)
    for at in {0, atoms // 2, atoms - 1}:
        for value in (-1, 4):
            bad = species.clone()
            bad[at] = value
            assert look(offsets, nbr, bad)[2]
            with pytest.raises(ValueError, match="species index"):
                validate_density_csr(offsets, nbr, atoms, edges, species=bad, species_count=4)
        bad = offsets.clone()
        bad[at] = edges + 1
        assert look(bad, nbr, species)[0]
        with pytest.raises(ValueError, match="row_offsets"):
            validate_density_csr(bad, nbr, atoms, edges)
    # the rows of centres: the offsets they came from
    centers = torch.repeat_interleave(torch.arange(atoms, device=gpu), offsets.diff())
    assert torch.equal(native.csr_offsets(centers, atoms), offsets)
    # what the device cannot look at: other layouts keep the Torch checks
    if edges > 1:
        strided = torch.stack([nbr, nbr], dim=1)[:, 0]
        assert native.check_indices((strided, 0, atoms, False)) is None
        assert validate_density_csr(offsets, strided, atoms, edges)
