"""The sorted factorized-angular kernels against the oracle, and the plans they leave to the others."""

import numpy as np
import pytest

import oracle
from tests._dag import random_dag
from tests._util import TOL, flush
from tests.test_gpu_factorized_angular import _args, _cplx_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float64", "complex64"])
@pytest.mark.parametrize("batch,sources,leaves,nodes", [
    (1, 1, (1, 1), 6), (63, 3, (1, 2, 1, 0), 12), (65, 5, (2, 2, 1), 20),
    (33, 40, (1, 0), 7),            # more sources than lanes a sample leaves room for
    (17, 2, (6, 6, 5, 4, 6, 6), 40),  # a wide workspace: few lanes a wave
])
@pytest.mark.parametrize("ordered", [True, False])
def test_sorted_plans_against_the_oracle(gpu, dtype, batch, sources, leaves, nodes, ordered):
    """Several sources a sample, runs of one and of many coefficients, and, unordered, a node that reads
    its child before the child is computed (zeros, as the reference's replay has it), or, where no later
    node can be that child, nodes whose values lie in another order."""
    flush(f"sorted factorized plan, {batch} x {sources}, {len(leaves)} leaves, {nodes} nodes, {dtype}, {ordered}")
    import torch

    from ye3t_amd.runtime import factorized_angular, native

    dt = getattr(torch, dtype)
    tables, S, D = random_dag(71 + nodes, complex_data=dt.is_complex, leaves_L=leaves, sources=sources, max_nodes=nodes)
    if not ordered:
        n = len(leaves)  # the first merge: a later node of as many components in its left child's place
        dims = tables["node_dimensions"]
        later = [k for k in range(n + 1, len(dims)) if dims[k] == dims[tables["node_left"][n]]]
        if later:
            tables["node_left"][n] = later[-1]
        else:
            offsets = tables["node_offsets"]  # of all but the last node, which ends the workspace
            offsets[:-1] = offsets[-1] - offsets[:-1] - dims[:-1]
    for k in ("coefficient_values", "projection_values"):
        tables[k] = torch.as_tensor(tables[k]).to(dt).numpy()
    rng = np.random.default_rng(nodes)
    draw = lambda *s: rng.normal(size=s) + (1j * rng.normal(size=s) if dt.is_complex else 0)  # noqa: E731
    x = torch.as_tensor(draw(batch, S * D), device=gpu).to(dt).requires_grad_(True)
    W = int(tables["node_offsets"][-1] + tables["node_dimensions"][-1])
    K = len(tables["root_nodes"]) * (len(tables["projection_values"]) // S) * 3
    out = factorized_angular(x, *_args(tables, gpu, dt), S, W, K)
    kind = "fa_sorted" if ordered else "fa"
    assert native.last_kernel() == f"{kind}_forward_kernel"
    xr = x.detach().cpu().numpy()
    tol = TOL["f64"] if dtype == "float64" else TOL["f32"]
    assert _cplx_err(out.detach().cpu().numpy(), oracle.factorized_angular(xr, tables, S)) < tol
    g = torch.as_tensor(draw(batch, K), device=gpu).to(dt)
    (gx,) = torch.autograd.grad(out, x, g)
    torch.cuda.synchronize()
    assert _cplx_err(gx.cpu().numpy(), oracle.factorized_angular_adjoint(g.cpu().numpy(), xr, tables, S)) < tol
