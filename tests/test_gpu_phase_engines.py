"""The CG engines behind the resident one: one workgroup per group of right-hand sides up to 32768 rows, a
launch per solver phase above, and the launch-per-phase engine of segmented solves. They run what
the resident engine does not take (rows longer than seven entries, systems beyond the register files)
and what it gives up on, so they are reached here in both ways: operators of nine entries per row, and
the large-system tests of test_gpu_solvers.py with teams that give up at once."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import test_gpu_solvers as solvers
from oracle import oracle as O
from test_gpu_resident import DEV, SHIFT, _check, _segmented, no_waiting, resident

pytestmark = pytest.mark.gpu


def _nine_point(nx, ny, shift=SHIFT):
    """Nine-point operator of an nx x ny grid, zero row sums plus a shift and noise on the diagonal (none with
    shift 0: singular)."""
    n = nx * ny
    idx = np.arange(n).reshape(ny, nx)
    rows, cols = [np.arange(n)], [np.arange(n)]
    for dy in (-1, 0, 1):
        for dx in (-1, 0, 1):
            if (dx, dy) == (0, 0):
                continue
            rows.append(idx[max(0, -dy):ny + min(0, -dy), max(0, -dx):nx + min(0, -dx)].ravel())
            cols.append(idx[max(0, dy):ny + min(0, dy), max(0, dx):nx + min(0, dx)].ravel())
    r, c = np.concatenate(rows), np.concatenate(cols)
    order = np.lexsort((c, r))
    r, c = r[order], c[order]
    row = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32)
    diag = np.bincount(r, minlength=n) - 1.0
    if shift:
        diag += shift + np.random.default_rng(n).uniform(0, 0.5, n)
    return row, c.astype(np.int32), np.where(r == c, diag[r], -1.0)


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("opts", [dict(), dict(residualResetSteps=7), dict(returnBestResult=True)],
                         ids=["plain", "reset", "best"])
@pytest.mark.parametrize("shape,nrhs", [((60, 50), 5), ((129, 255), 1), ((220, 170), 1), ((181, 183), 6)])
def test_nine_entries_per_row(shape, nrhs, opts, dtype):
    print(f"[phase engines] {shape} x {nrhs} {opts} {np.dtype(dtype).name}", flush=True)
    _check(*_nine_point(*shape), nrhs, dtype, engine={}, **opts)


@pytest.mark.parametrize("case", ["cg-f64", "cg-f32", "ill-conditioned", "contract", "projected-f64", "projected-f32",
                                  "ell-copy", "zero-rhs", "jacobi-f64", "jacobi-f32"])
def test_large_system_tests_with_teams_that_give_up(case):
    import phipict_amd as pa
    from phipict_amd import profiling

    name, _, dt = case.partition("-f")
    dtype = np.float32 if dt == "32" else np.float64
    before = profiling.resident_counts()
    try:
        with no_waiting():
            {"cg": lambda: solvers.test_cg_matches_oracle("large", dtype),
             "ill-conditioned": lambda: solvers.test_ill_conditioned_large_solve(False),
             "contract": lambda: solvers.test_result_contract_edge_cases("large"),
             "projected": lambda: solvers.test_singular_cg_projected("large", dtype),
             "ell-copy": lambda: solvers.test_ell_copy_gives_identical_solves(False),
             "zero-rhs": lambda: solvers.test_zero_rhs_shortcut_on_device(False),
             "jacobi": lambda: solvers.test_jacobi_preconditioned_matches_oracle(pa, "large", False, dtype)}[name]()
    finally:
        pa.SetKrylovSettings()
    finished, declined, gave_up = (b - a for a, b in zip(before, profiling.resident_counts()))
    assert finished == 0 and declined == 0 and gave_up > 0


SIZES = [(24, 16), (40, 20), (90, 70), (48, 24), (20, 28), (7, 5)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("tile_rows", [256, 1024, 4096])
def test_segmented_nine_entries_per_row(tile_rows, dtype):
    import phipict_amd as pa

    parts = [_nine_point(*s) for s in SIZES]
    segs = np.concatenate([[0], np.cumsum([p[0].size - 1 for p in parts])])
    n, S, ncomp = int(segs[-1]), len(parts), 2
    tol = 1e-9 if dtype == np.float64 else 1e-4
    tdt = torch.float64 if dtype == np.float64 else torch.float32
    rng = np.random.default_rng(5)
    b = rng.standard_normal((ncomp, n)).astype(dtype)
    x0 = (0.1 * rng.standard_normal((ncomp, n))).astype(dtype)
    b[1, segs[2]:segs[3]] = 0.0  # one piece with an exactly zero right-hand side
    A = _segmented([(r, c, v.astype(dtype)) for r, c, v in parts], segs)
    x = torch.as_tensor(x0.reshape(-1).copy(), device=DEV)
    assert A.getDtype() == tdt
    with resident():
        infos = pa.SolveSegmented(A, segs.tolist(), torch.as_tensor(b.reshape(-1), device=DEV), x, maxIterations=4000,
                                  tolerance=tol, tileRows=tile_rows)
    xs = x.cpu().numpy().reshape(ncomp, n)
    for c in range(ncomp):
        for s, (lo, hi) in enumerate(zip(segs[:-1], segs[1:])):
            info = infos[c * S + s]
            if not b[c, lo:hi].any():
                assert info.converged and info.usedIterations == 0 and not xs[c, lo:hi].any()
                continue
            xo = x0[c, lo:hi].copy()
            r_, c_, v_ = parts[s]
            ref = O.cg(r_, c_, v_.astype(dtype), b[c, lo:hi].copy(), xo, tol, maxit=4000)
            assert info.converged and ref.converged
            assert abs(info.usedIterations - ref.used_iterations) <= (1 if dtype == np.float64 else 4)
            bound = 2 * np.sqrt(hi - lo) * tol / SHIFT + np.finfo(dtype).eps * 64 * np.linalg.norm(xo)
            assert np.linalg.norm(xs[c, lo:hi].astype(np.float64) - xo.astype(np.float64)) <= bound


def test_segmented_projected_nine_entries_and_captured_chunks():
    """Singular pieces with right-hand sides of nonzero mean, from direct launches and from captured chunks of
    iterations: the same bits, and the oracle's solution up to the constant."""
    import phipict_amd as pa

    parts = [_nine_point(*s, shift=0) for s in SIZES]
    segs = np.concatenate([[0], np.cumsum([p[0].size - 1 for p in parts])])
    b = np.random.default_rng(6).standard_normal(segs[-1]) + 0.3
    A, bt = _segmented(parts, segs), torch.as_tensor(b, device=DEV)
    runs = {}
    try:
        for graphs in (False, True):
            pa.SetKrylovSettings(useGraphs=graphs)
            outs = []
            for _ in range(3):
                x = torch.zeros_like(bt)
                with resident():
                    infos = pa.SolveSegmented(A, segs.tolist(), bt, x, maxIterations=4000, tolerance=1e-9,
                                              matrixRankDeficient=True)
                outs.append((x.clone(), [(i.usedIterations, i.finalResidual, i.converged) for i in infos]))
            runs[graphs] = outs
    finally:
        pa.SetKrylovSettings()
    for (xa, ia), (xb, ib) in zip(runs[False], runs[True]):
        assert ia == ib and torch.equal(xa, xb)
    xs = runs[False][0][0].cpu().numpy()
    for s, (lo, hi) in enumerate(zip(segs[:-1], segs[1:])):
        r_, c_, v_ = parts[s]
        xo = np.zeros(hi - lo)
        ref = O.cg(r_, c_, v_, b[lo:hi].copy(), xo, 1e-9, maxit=4000, project=True)
        used, _, converged = runs[False][0][1][s]
        assert converged and ref.converged and abs(used - ref.used_iterations) <= 1
        # both residuals are below tol sqrt(n); the smallest nonzero eigenvalue of the nine-point operator of an
        # nx x ny grid is above that of the five-point one, 4 sin^2(pi / (2 max(nx, ny)))
        lam = 4 * np.sin(np.pi / (2 * max(SIZES[s]))) ** 2
        d = (xs[lo:hi] - xs[lo:hi].mean()) - (xo - xo.mean())
        assert np.linalg.norm(d) <= 2 * 1.1 * np.sqrt(hi - lo) * 1e-9 / lam
