"""AMG-PCG where the workgroups of its finest-level kernels change: one row less, equal to and one more than
a workgroup of 1024 rows, a last workgroup of one wavefront, and one and three right-hand sides.

Tolerance: a solve stops once the recurrence's residual is below tol in the normalised 2-norm; the operator's
smallest eigenvalue is at least the shift, so the solution is within sqrt(n) tol / shift of the exact one, and the
true residual follows the recurrence's within a few ulp of |A| |x| per iteration (a tenth of tol here)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
SHIFT = 0.05


@pytest.mark.parametrize("nrhs", [1, 3])
@pytest.mark.parametrize("shape", [(33, 31), (32, 32), (41, 25), (52, 40), (128, 65)])
def test_amg_pcg_workgroup_edges(shape, nrhs):
    print(f"[pcg shapes] {shape} x{nrhs}", flush=True)
    import scipy.sparse as sp
    import scipy.sparse.linalg as spl

    import phipict_amd as pa
    from phipict_amd.solvers import amg

    one = [sp.diags([-np.ones(k - 1), 2 * np.ones(k), -np.ones(k - 1)], [-1, 0, 1]) for k in shape]
    M = (sp.kron(one[0], sp.eye(shape[1])) + sp.kron(sp.eye(shape[0]), one[1]) + SHIFT * sp.eye(shape[0] * shape[1])).tocsr()
    M.sort_indices()
    n = M.shape[0]
    A = pa.CSRmatrix(torch.as_tensor(M.data, device=DEV), torch.as_tensor(M.indices.astype(np.int32), device=DEV),
                     torch.as_tensor(M.indptr.astype(np.int32), device=DEV))
    h = amg.build_amg_hierarchy(A, project_constant=False, native_dtype=torch.float32)
    b = np.random.default_rng(n + nrhs).standard_normal((nrhs, n))
    x = torch.zeros(nrhs * n, dtype=torch.float64, device=DEV)
    tol = 1e-9
    infos = amg.amg_pcg_solve(torch.as_tensor(b.ravel(), device=DEV), x, h, tol=tol, max_iter=200)
    assert len(infos) == nrhs and all(i.converged for i in infos)
    xs = x.cpu().numpy().reshape(nrhs, n)
    for k in range(nrhs):
        assert np.linalg.norm(b[k] - M @ xs[k]) <= 1.1 * tol * np.sqrt(n)
        assert np.linalg.norm(xs[k] - spl.spsolve(M.tocsc(), b[k])) <= 1.1 * tol * np.sqrt(n) / SHIFT
