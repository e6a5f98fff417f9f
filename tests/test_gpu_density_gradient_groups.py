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


def _error(got, ref):
    """The three edges below epsilon are larger than the others by their 1 / epsilon, and a root mean square over
    all E edges is sqrt(E / 3) below theirs: each part by itself."""
    return max(column_rel_error(got[:3], ref[:3]), column_rel_error(got[3:], ref[3:]))


@pytest.mark.parametrize("mode,channels,dtypes", [("single", 1, ("f64", "f64")), ("species", 3, ("f32", "f64"))])
@pytest.mark.parametrize("n_max", [0, 1])
@pytest.mark.parametrize("lam", [0.0, 800.0])
def test_rows_that_lambda_does_not_enter(gpu, mode, channels, dtypes, n_max, lam):
    """R_0 and R_1 hold no lambda: where expm1(lambda) is zero or infinite, and higher rows are no numbers,
    a model of those two rows has the gradient it always had."""
    flush(f"grouped edge gradient {mode} x{channels}, n_max {n_max}, lambda {lam}, {dtypes}")
    import torch

    from ye3t_amd.runtime import native

    inp = _workload(mode, 1500, 100, 93, n_max, 4, channels)
    inp["lambda"] = lam
    gA = np.random.default_rng(94).normal(size=(1500, channels, n_max + 1, 25))
    d, kw = _device(inp, dtypes[0], gpu)
    gd = torch.as_tensor(gA, device=gpu)
    got = native.ace_density_edge_gradient(gd, d["edge_vectors"], d["row_offsets"], d["neighbors"], **kw)
    ref = oracle.ace_density_edge_gradient(rounded_inputs(inp, dtypes[0]), gA)
    assert inp["edge_count"] >= 65536
    got = got.cpu().numpy()
    err = _error(got, ref)
    flush(f"  {err:.2e}")
    assert np.isfinite(ref).all() and err < TOL[dtypes[0]]


@pytest.mark.parametrize("mode,channels", [("single", 1), ("species", 3)])
@pytest.mark.parametrize("degrees", ["one atom", "first tenth", "last atoms", "far apart", "few atoms", "rising"])
def test_uneven_structures(gpu, mode, channels, degrees):
    """Shares of the work that begin and end within atoms, runs of empty atoms longer than a chunk's window at
    the start, between and at the end, and atoms of many chunks."""
    flush(f"grouped edge gradient {mode} x{channels}, {degrees}")
    import torch

    from ye3t_amd.runtime import native

    rng = np.random.default_rng(95)
    counts = {"one atom": [100003], "first tenth": [230] * 450 + [0] * 4050, "last atoms": [0] * 5000 + [337] * 297,
              "far apart": np.where(np.arange(5000) % 50 == 7, 1009, 0), "few atoms": [701] * 143,
              "rising": np.arange(1800) // 16}[degrees]
    inp = _workload(mode, len(counts), 1, 96, 15, 6, channels)
    E = int(np.sum(counts))
    vec = rng.normal(size=(E, 3))
    inp.update(edge_count=E, centers=np.repeat(np.arange(len(counts)), counts),
               row_offsets=np.concatenate([[0], np.cumsum(counts)]).astype(np.int64),
               neighbors=rng.integers(0, len(counts), E),
               edge_vectors=vec / np.linalg.norm(vec, axis=1, keepdims=True) * rng.uniform(0.05, 5.3, (E, 1)))
    gA = rng.normal(size=(len(counts), channels, 16, 49))
    d, kw = _device(inp, "f64", gpu)
    got = native.ace_density_edge_gradient(torch.as_tensor(gA, device=gpu), d["edge_vectors"], d["row_offsets"],
                                           d["neighbors"], **kw)
    assert native.last_kernel() == "density_edge_gradient_mfma_kernel"
    err = column_rel_error(got.cpu().numpy(), oracle.ace_density_edge_gradient(inp, gA))
    flush(f"  {err:.2e}")
    assert err < TOL["f64"]


@pytest.mark.parametrize("channels,dtypes", [(1, ("f64", "f64")), (3, ("f32", "f64")), (2, ("f32", "f32"))])
@pytest.mark.parametrize("n_max", [6, 7, 8, 10, 11, 12, 13, 15])
def test_radial_rows(gpu, n_max, channels, dtypes):
    """Every count of compiled radial rows, filled and in part."""
    flush(f"grouped edge gradient, {channels} channels, n_max {n_max}, {dtypes}")
    import torch

    from ye3t_amd.runtime import native

    inp = _workload("species" if channels > 1 else "single", 4500 if channels == 1 else 1500, 100, 97, n_max, 6, channels)
    shape = (inp["atom_count"], channels, n_max + 1, 49)
    d, kw = _device(inp, dtypes[0], gpu)
    gd = torch.as_tensor(np.random.default_rng(98).normal(size=shape), device=gpu)
    gd = gd.to(torch.float64 if dtypes[1] == "f64" else torch.float32)
    got = native.ace_density_edge_gradient(gd, d["edge_vectors"], d["row_offsets"], d["neighbors"], **kw).cpu().numpy()
    assert native.last_kernel() == "density_edge_gradient_mfma_kernel"
    ref = oracle.ace_density_edge_gradient(rounded_inputs(inp, dtypes[0]), gd.double().cpu().numpy())
    err = _error(got, ref)
    flush(f"  {err:.2e}")
    assert err < TOL[dtypes[0]]


@pytest.mark.parametrize("channels,atoms,degree,n_max,l_max,grouped", [
    (2, 3000, 60, 6, 6, True), (2, 3000, 60, 5, 6, False),       # seven radial rows, six
    (4, 4500, 36, 12, 4, True), (5, 4500, 36, 12, 4, False),     # four edges a group and above, below
    (2, 2200, 60, 15, 4, True), (2, 2150, 60, 15, 4, False),     # 65 536 edges, fewer
    (1, 2200, 150, 9, 6, True), (1, 2200, 150, 8, 6, False),     # one channel: 7.5e7 values to gather, fewer
    (2, 2300, 60, 14, 4, True), (2, 2300, 60, 13, 4, False),     # 2.5e7 of them, fewer
    (2, 3500, 60, 15, 3, False), (2, 2300, 60, 15, 7, False),    # l_max
])
def test_both_sides_of_the_rule(gpu, channels, atoms, degree, n_max, l_max, grouped):
    """The kernel that a call goes to at each line of the rule, and its values there."""
    flush(f"edge gradient rule: {channels} channels, {atoms} x {degree}, n_max {n_max}, l_max {l_max}")
    import torch

    from ye3t_amd.runtime import native

    inp = _workload("species" if channels > 1 else "single", atoms, 0, 99, n_max, l_max, channels)
    rng = np.random.default_rng(100)
    E = atoms * degree // 2
    vec = rng.normal(size=(E, 3))
    counts = np.full(atoms, degree // 2)
    inp.update(edge_count=E, centers=np.repeat(np.arange(atoms), counts),
               row_offsets=np.concatenate([[0], np.cumsum(counts)]).astype(np.int64),
               neighbors=rng.integers(0, atoms, E),
               edge_vectors=vec / np.linalg.norm(vec, axis=1, keepdims=True) * rng.uniform(0.5, 5.3, (E, 1)))
    gA = rng.normal(size=(atoms, channels, n_max + 1, (l_max + 1) ** 2))
    d, kw = _device(inp, "f64", gpu)
    got = native.ace_density_edge_gradient(torch.as_tensor(gA, device=gpu), d["edge_vectors"], d["row_offsets"],
                                           d["neighbors"], **kw)
    assert native.last_kernel() == ("density_edge_gradient_mfma_kernel" if grouped else "density_edge_gradient_kernel")
    assert column_rel_error(got.cpu().numpy(), oracle.ace_density_edge_gradient(inp, gA)) < TOL["f64"]
