"""The bounds of a neighbour list's positions against Torch's, and what is not a number in them."""

import ctypes
import math

import pytest

from tests._util import flush

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float64", "float32"])
@pytest.mark.parametrize("atoms", [1, 63, 257, 16384, 40001])
def test_bounds(gpu, dtype, atoms):
    flush(f"position bounds, {atoms} atoms, {dtype}")
    import torch

    from ye3t_amd.runtime import native, neighbor_list

    pos = torch.randn((atoms, 3), generator=torch.Generator().manual_seed(atoms), dtype=torch.float64)
    pos = pos.to(gpu, getattr(torch, dtype))

    def bounds(p):
        out = (ctypes.c_double * 6)()
        code = native.F64 if dtype == "float64" else native.F32
        assert native.lib().ye3t_hip_position_bounds(code, p.data_ptr(), atoms, out, native._stream()) == 0
        return list(out)

    lo, hi = torch.aminmax(pos, dim=0)
    assert bounds(pos) == lo.double().tolist() + hi.double().tolist()
    for at in {0, atoms // 2, atoms - 1}:
        for value in (math.nan, math.inf, -math.inf):
            bad = pos.clone()
            bad[at, 1] = value
            b = bounds(bad)
            assert not (math.isfinite(b[1]) and math.isfinite(b[4]))
            with pytest.raises(ValueError, match="finite"):
                neighbor_list(bad, 1.0)
