"""The grouped (matrix-core) edge gradient against the oracle."""

import numpy as np
import pytest

import oracle
from tests._util import TOL, column_rel_error, flush, rounded_inputs
from tests.test_gpu_density_gradient import _device, _workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,channels,atoms,degree,n_max,l_max,dtypes", [
    ("single", 1, 1100, 150, 8, 4, ("f64", "f64")),     # one group an atom, atoms of several windows
    ("species", 3, 5000, 40, 10, 4, ("f64", "f64")),    # 11 radial rows
    ("species", 7, 1500, 130, 15, 5, ("f32", "f64")),   # 16 radial rows, long and short groups
    ("species", 2, 40000, 4, 3, 6, ("f32", "f32")),     # below four edges a group: the other kernel
    ("species", 2, 9000, 18, 3, 6, ("f32", "f32")),     # four rows of nine compiled, many atoms a chunk
    ("species", 8, 1800, 96, 12, 6, ("f64", "f64")),
])
def test_grouped_edge_gradient(gpu, mode, channels, atoms, degree, n_max, l_max, dtypes):
    """Ragged rows with empty atoms, atoms of more than 64 edges, edges beyond the cutoff and below epsilon."""
    flush(f"grouped edge gradient {mode} x{channels}, n_max {n_max}, l_max {l_max}, {dtypes}")
    import torch

    from ye3t_amd.runtime import native

    dtype, adjoint = dtypes
    inp = _workload(mode, atoms, degree, 91, n_max, l_max, channels)
    rng = np.random.default_rng(92)
    gA = rng.normal(size=(atoms, channels, n_max + 1, (l_max + 1) ** 2))
    d, kw = _device(inp, dtype, gpu)
    gd = torch.as_tensor(gA, device=gpu).to(torch.float64 if adjoint == "f64" else torch.float32)
    got = native.ace_density_edge_gradient(gd, d["edge_vectors"], d["row_offsets"], d["neighbors"], **kw)
    ref = oracle.ace_density_edge_gradient(rounded_inputs(inp, dtype), gd.double().cpu().numpy())
    got = got.cpu().numpy()
    # the three edges below epsilon are larger by their 1 / epsilon: the others by themselves too
    err = max(column_rel_error(got, ref), column_rel_error(got[3:], ref[3:]))
    assert inp["edge_count"] >= 65536
    flush(f"  {err:.2e}")
    assert err < (TOL["f64"] if dtype == "f64" else TOL["f32"])
