"""The resident CG engine against the oracle where its shapes change: one workgroup up to the rows its
registers hold (4096 with five entries per row, 3072 with seven), teams of 512-thread workgroups with
one, two and four rows per thread, more right-hand sides than run at once, rows longer than the
kernels take (handed to the other engines).

Tolerances: the engine sums in another order than the oracle, so a solve may stop an iteration
earlier or later; the solutions then differ by what the stopping residual leaves open, which for these
shifted operators (smallest eigenvalue >= shift) is at most sqrt(n) tol / shift in the 2-norm.

Every test states which engine the solve came from, by the library's counts of resident solves finished,
declined and given up."""
from __future__ import annotations

from contextlib import contextmanager

import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda", 0)
SHIFT = 0.05


def _grid_operator(shape, extra=None):
    """2d + 1 point operator of a grid with Dirichlet walls, diagonal 2d + SHIFT + noise; ``extra``: pairs of
    rows coupled besides."""
    n, d = int(np.prod(shape)), len(shape)
    idx = np.arange(n).reshape(shape)
    rows, cols = [np.arange(n)], [np.arange(n)]
    for ax in range(d):
        lo, hi = np.moveaxis(idx, ax, 0)[:-1].ravel(), np.moveaxis(idx, ax, 0)[1:].ravel()
        rows += [lo, hi]
        cols += [hi, lo]
    for i, j in extra or []:
        rows += [np.array([i, j])]
        cols += [np.array([j, i])]
    r, c = np.concatenate(rows), np.concatenate(cols)
    order = np.lexsort((c, r))
    r, c = r[order], c[order]
    row = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))]).astype(np.int32)
    off = np.bincount(r, minlength=n) - 1
    diag = np.maximum(2 * d, off) + SHIFT + np.random.default_rng(n).uniform(0, 0.5, n)
    return row, c.astype(np.int32), np.where(r == c, diag[r], -1.0)


@contextmanager
def resident(finished=0, declined=0, gave_up=0):
    """The solves inside went to the resident engine this often, with these outcomes."""
    from phipict_amd import profiling

    before = profiling.resident_counts()
    yield
    got = tuple(b - a for a, b in zip(before, profiling.resident_counts()))
    assert got == (finished, declined, gave_up), got


def _check(row, col, val, nrhs, dtype, engine=dict(finished=1), **opts):
    import phipict_amd as pa

    n = row.size - 1
    f64 = dtype == np.float64
    tol = 1e-9 if f64 else 1e-4
    b = np.random.default_rng(7).standard_normal(nrhs * n).astype(dtype)
    x0 = (0.1 * np.random.default_rng(8).standard_normal(nrhs * n)).astype(dtype)
    tdt = torch.float64 if f64 else torch.float32
    A = pa.CSRmatrix(torch.as_tensor(val, dtype=tdt, device=DEV), torch.as_tensor(col, device=DEV),
                     torch.as_tensor(row, device=DEV))
    x = torch.as_tensor(x0.copy(), device=DEV)
    with resident(**engine):
        infos = pa.SolveLinear(A, torch.as_tensor(b, device=DEV), x, maxIterations=4000, tolerance=tol, **opts)
    xs = x.cpu().numpy().reshape(nrhs, n)
    for k in sorted({0, nrhs - 1}):
        xo = x0[k * n:(k + 1) * n].copy()
        ref = O.cg(row, col, val.astype(dtype), b[k * n:(k + 1) * n].copy(), xo, tol, maxit=4000,
                   reset_every=opts.get("residualResetSteps", 0), return_best=opts.get("returnBestResult", False))
        assert infos[k].converged and ref.converged
        assert abs(infos[k].usedIterations - ref.used_iterations) <= (1 if f64 else 4)
        bound = 2 * np.sqrt(n) * tol / SHIFT + np.finfo(dtype).eps * 64 * np.linalg.norm(xo)
        assert np.linalg.norm(xs[k].astype(np.float64) - xo.astype(np.float64)) <= bound, (k, infos[k], ref)


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape,nrhs", [
    ((3, 1), 1), ((63, 65), 2), ((64, 64), 1), ((17, 241), 1),  # one workgroup to its last row, then a team
    ((12, 16, 16), 1), ((7, 439), 3),                           # 3072 and 3073 rows
    ((512, 256), 1), ((331, 396), 1),                           # 131072 rows on 256 workgroups, then two rows a thread
    ((40, 50, 60), 2), ((71, 60, 62), 1),                       # two teams at once; 264120 rows: four rows a thread
    ((120, 150), 40),                                           # more teams than run at once
])
def test_resident_cg_matches_oracle(shape, nrhs, dtype):
    print(f"[resident] {shape} x {nrhs} {np.dtype(dtype).name}", flush=True)
    _check(*_grid_operator(shape), nrhs, dtype)


@pytest.mark.parametrize("opts", [dict(residualResetSteps=5), dict(returnBestResult=True)], ids=["reset", "best"])
@pytest.mark.parametrize("shape", [(30, 41), (20, 31, 33)], ids=["workgroup", "team"])
def test_resident_cg_options(shape, opts):
    _check(*_grid_operator(shape), 2, np.float64, **opts)


@pytest.mark.parametrize("shape", [(512, 256), (331, 396), (71, 60, 62)], ids=["256x1", "129x2", "129x4"])
def test_residual_replacement_in_large_teams(shape):
    """Teams whose members poll the sums in two rounds (more than 128 workgroups), with one, two and four rows
    per thread: replacements exchange x between members that are not neighbours of each other's rows."""
    print(f"[resident] replacement {shape}", flush=True)
    _check(*_grid_operator(shape), 1, np.float64, residualResetSteps=7)


def test_batch_of_more_values_than_32_bits_count():
    """2^31 + 2^20 values in right-hand sides of 4096 rows, one workgroup each: offsets into the vectors."""
    import phipict_amd as pa

    row, col, val = _grid_operator((64, 64))
    val = np.where(val > 0, val + 16.0, val)
    n, nrhs = 4096, (1 << 19) + 256
    print(f"[resident] {nrhs} right-hand sides of {n} rows f32", flush=True)
    A = pa.CSRmatrix(torch.as_tensor(val, dtype=torch.float32, device=DEV), torch.as_tensor(col, device=DEV),
                     torch.as_tensor(row, device=DEV))
    b = torch.empty(nrhs * n, dtype=torch.float32, device=DEV)
    b.normal_(generator=torch.Generator(DEV).manual_seed(3))
    x = torch.zeros_like(b)
    try:
        with resident(finished=1):
            infos = pa.SolveLinear(A, b, x, maxIterations=100, tolerance=1e-4)
        assert all(i.converged for i in infos)
        r = np.repeat(np.arange(n), np.diff(row))
        for k in (0, (1 << 19) - 1, 1 << 19, nrhs - 1):
            xk, bk = (v[k * n:(k + 1) * n].cpu().numpy().astype(np.float64) for v in (x, b))
            res = bk - np.bincount(r, weights=val * xk[col], minlength=n)
            # the stopping residual, and the rounding of FP32 in sums of ~40 |x|
            assert np.linalg.norm(res) <= np.sqrt(n) * 1e-4 + 40 * 8 * np.finfo(np.float32).eps * np.linalg.norm(xk), k
    finally:
        del b, x
        pa.ReleaseKrylovWorkspaces()
        torch.cuda.empty_cache()


def test_threads_do_not_wait_for_each_others_queued_work():
    """A thread with a second of products queued on its stream before its solve, and a thread that solves
    meanwhile on another: the second is done long before the first one's queue is. Then both solve at once,
    over and over, in teams that fit the device together and teams that do not."""
    import threading

    import phipict_amd as pa
    from phipict_amd import profiling

    def system(shape):
        row, col, val = _grid_operator(shape)
        n = row.size - 1
        A = pa.CSRmatrix(*(torch.as_tensor(a, device=DEV) for a in (val, col, row)))
        b = torch.as_tensor(np.random.default_rng(n).standard_normal(n), device=DEV)
        x = torch.zeros(n, dtype=torch.float64, device=DEV)
        ref = torch.zeros_like(x)
        pa.SolveLinear(A, b, ref, maxIterations=4000, tolerance=1e-9)
        return A, b, x, ref

    def solve(s):
        A, b, x, ref = s
        x.zero_()
        info = pa.SolveLinear(A, b, x, maxIterations=4000, tolerance=1e-9)[0]
        assert info.converged and torch.equal(x, ref)

    small = [system((70, 65)), system((90, 70))]
    large = [system((400, 200)), system((300, 290))]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    m = torch.randn(2048, 2048, device=DEV)
    out = torch.empty_like(m)
    queued, end = threading.Event(), torch.cuda.Event()
    seen, counts, errors = {}, [None, None], []
    line = threading.Barrier(2, timeout=60)

    def run(me):
        try:
            before = profiling.resident_counts()
            with torch.cuda.stream(streams[me]):
                solve(small[me])  # both threads have their workspaces
                line.wait()
                if me == 0:
                    for _ in range(6000):
                        torch.mm(m, m, out=out)
                    end.record()
                    queued.set()
                    solve(small[0])
                else:
                    queued.wait(60)
                    solve(small[1])
                    seen["busy"] = not end.query()
                line.wait()
                for s in (small[me], large[me]) * 20:
                    solve(s)
            counts[me] = tuple(b - a for a, b in zip(before, profiling.resident_counts()))
        except BaseException as e:  # reported below, in the test's own thread
            errors.append(e)
            line.abort()

    threads = [threading.Thread(target=run, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    assert not errors, errors
    assert seen["busy"]
    assert counts == [(42, 0, 0)] * 2


def test_zero_right_hand_sides_of_a_batch():
    """All zero: x = 0 without iterating, from any start guess. Some zero: solved as any other, from the start
    guess, with the oracle's iterations."""
    import phipict_amd as pa
    from phipict_amd import profiling

    row, col, val = _grid_operator((200, 200))
    n, nrhs, tol = 40000, 3, 1e-9
    A = pa.CSRmatrix(*(torch.as_tensor(a, device=DEV) for a in (val, col, row)))
    x0 = 1.0 + 0.1 * np.random.default_rng(3).standard_normal(nrhs * n)
    x = torch.as_tensor(x0.copy(), device=DEV)
    profiling.start(1)
    try:
        with resident(finished=1):
            infos = pa.SolveLinear(A, torch.zeros_like(x), x, maxIterations=4000, tolerance=tol)
    finally:
        profiling.stop()
    assert all(i.converged and i.usedIterations == 0 for i in infos) and not x.any()
    # one opening, where solving the three takes about fifty iterations of 5 us
    assert sum(t.sampled_ms for t in profiling.read() if t.name == "cg_small") < 0.1
    b = np.zeros(nrhs * n)
    b[n:2 * n] = np.random.default_rng(4).standard_normal(n)
    x = torch.as_tensor(x0.copy(), device=DEV)
    with resident(finished=1):
        infos = pa.SolveLinear(A, torch.as_tensor(b, device=DEV), x, maxIterations=4000, tolerance=tol)
    for k in range(nrhs):
        xo = x0[k * n:(k + 1) * n].copy()
        ref = O.cg(row, col, val, b[k * n:(k + 1) * n].copy(), xo, tol, maxit=4000)
        assert infos[k].converged and abs(infos[k].usedIterations - ref.used_iterations) <= 1 and ref.used_iterations > 10
        assert np.linalg.norm(x[k * n:(k + 1) * n].cpu().numpy() - xo) <= 2 * np.sqrt(n) * tol / SHIFT


@contextmanager
def no_waiting():
    """Teams of several workgroups give up at the first word that is not there yet."""
    from phipict_amd import _lib

    _lib.call("pp_resident_wait", 0)
    try:
        yield
    finally:
        _lib.call("pp_resident_wait", -1)


@pytest.mark.parametrize("dtype", [np.float64, np.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("shape,nrhs", [((65, 64), 3), ((200, 190), 2), ((331, 396), 1), ((20, 31, 33), 2), ((71, 60, 62), 1)])
def test_given_up_solves_are_run_by_the_other_engines(shape, nrhs, dtype):
    """Rows up to 32768: the one-workgroup engine; above: a launch per phase."""
    print(f"[resident] giving up {shape} x {nrhs} {np.dtype(dtype).name}", flush=True)
    with no_waiting():
        _check(*_grid_operator(shape), nrhs, dtype, engine=dict(gave_up=1))


@pytest.mark.parametrize("n", [2000, 9000])
def test_rows_beyond_the_kernels_take_another_engine(n):
    """One row of 13 entries among rows of five: no rows dropped."""
    _check(*_grid_operator((n // 50, 50), extra=[(0, n - 1 - 7 * k) for k in range(10)]), 1, np.float64,
           engine=dict(declined=1))


def test_a_declined_solve_leaves_nothing_behind():
    """The words by which a launch reports are not taken for those of a solve before, also where the workspace
    was released and its memory comes back as it was."""
    import phipict_amd as pa

    for shape in ((40, 50), (180, 50)):
        pa.ReleaseKrylovWorkspaces()
        _check(*_grid_operator(shape, extra=[(0, 1990 - 7 * k) for k in range(10)]), 1, np.float64, engine=dict(declined=1))
        pa.ReleaseKrylovWorkspaces()
        _check(*_grid_operator(shape), 1, np.float64)


def _segmented(parts, segs):
    import phipict_amd as pa

    offs = np.concatenate([[0], np.cumsum([p[1].size for p in parts])])
    row = np.concatenate([[0]] + [p[0][1:] + off for p, off in zip(parts, offs)]).astype(np.int32)
    col = np.concatenate([p[1] + o for p, o in zip(parts, segs)]).astype(np.int32)
    val = np.concatenate([p[2] for p in parts])
    return pa.CSRmatrix(*(torch.as_tensor(a, device=DEV) for a in (val, col, row)))


def _solve_pieces_from_the_start_guess(parts, engine):
    """Every piece is solved once, from the caller's start guess: the oracle's iterations."""
    import phipict_amd as pa

    segs = np.concatenate([[0], np.cumsum([p[0].size - 1 for p in parts])])
    rng = np.random.default_rng(12)
    b, x0 = rng.standard_normal(segs[-1]), 0.1 * rng.standard_normal(segs[-1])
    x = torch.as_tensor(x0.copy(), device=DEV)
    with resident(**engine):
        infos = pa.SolveSegmented(_segmented(parts, segs), segs.tolist(), torch.as_tensor(b, device=DEV), x,
                                  maxIterations=4000, tolerance=1e-9)
    xs = x.cpu().numpy()
    for k, (lo, hi) in enumerate(zip(segs[:-1], segs[1:])):
        xo = x0[lo:hi].copy()
        ref = O.cg(*parts[k], b[lo:hi].copy(), xo, 1e-9, maxit=4000)
        assert infos[k].converged and abs(infos[k].usedIterations - ref.used_iterations) <= 1, (k, infos[k], ref)
        assert np.linalg.norm(xs[lo:hi] - xo) <= 2 * np.sqrt(hi - lo) * 1e-9 / SHIFT + 1e-14 * np.linalg.norm(xo)


def test_giving_up_leaves_no_piece_half_solved():
    """The piece of several workgroups gives up, those of one workgroup beside it finish: all solved from the
    start guess."""
    with no_waiting():
        _solve_pieces_from_the_start_guess([_grid_operator((20, 31)), _grid_operator((70, 65)), _grid_operator((9, 40))],
                                           dict(gave_up=1))


def test_one_long_row_leaves_no_piece_half_solved():
    """A piece with a row of 13 entries among pieces of five: declined before any piece is solved."""
    _solve_pieces_from_the_start_guess([_grid_operator((20, 31)), _grid_operator((70, 65)), _grid_operator((9, 40)),
                                        _grid_operator((30, 20), extra=[(0, 599 - 7 * k) for k in range(10)])],
                                       dict(declined=1))


@pytest.mark.parametrize("shapes,ncomp", [
    ([(9, 7), (64, 64), (30, 2)], 2),                     # one workgroup each
    ([(65, 64), (20, 11), (300, 220), (3, 3)], 1),        # teams, the small ones beside them
    ([(420, 400)] * 3 + [(200, 150), (31, 17)], 1),       # 504 k rows: several launches
    ([(14, 15, 16), (33, 31, 30), (8, 9, 10)], 2),        # seven entries per row
], ids=["local", "mixed", "launches", "3d"])
def test_resident_segmented_cg_matches_oracle(shapes, ncomp):
    import phipict_amd as pa

    parts = [_grid_operator(s) for s in shapes]
    segs = np.concatenate([[0], np.cumsum([p[0].size - 1 for p in parts])])
    row = np.concatenate([[0]] + [p[0][1:] + off for p, off in
                                  zip(parts, np.concatenate([[0], np.cumsum([p[1].size for p in parts])]))]).astype(np.int32)
    col = np.concatenate([p[1] + o for p, o in zip(parts, segs)]).astype(np.int32)
    val = np.concatenate([p[2] for p in parts])
    n, S, tol = int(segs[-1]), len(shapes), 1e-9
    rng = np.random.default_rng(11)
    b, x0 = rng.standard_normal((ncomp, n)), 0.1 * rng.standard_normal((ncomp, n))
    b[0, segs[1]:segs[2]] = 0.0  # a zero right-hand side: x = 0, no iterations
    A = pa.CSRmatrix(*(torch.as_tensor(a, device=DEV) for a in (val, col, row)))
    x = torch.as_tensor(x0.reshape(-1).copy(), device=DEV)
    with resident(finished=1):
        infos = pa.SolveSegmented(A, segs.tolist(), torch.as_tensor(b.reshape(-1), device=DEV), x, maxIterations=4000,
                                  tolerance=tol)
    xs = x.cpu().numpy().reshape(ncomp, n)
    for c in range(ncomp):
        for s in range(S):
            lo, hi = int(segs[s]), int(segs[s + 1])
            info = infos[c * S + s]
            if not b[c, lo:hi].any():
                assert info.converged and info.usedIterations == 0 and not xs[c, lo:hi].any()
                continue
            xo = x0[c, lo:hi].copy()
            ref = O.cg(*parts[s], b[c, lo:hi].copy(), xo, tol, maxit=4000)
            assert info.converged and abs(info.usedIterations - ref.used_iterations) <= 1
            assert np.linalg.norm(xs[c, lo:hi] - xo) <= 2 * np.sqrt(hi - lo) * tol / SHIFT + 1e-14 * np.linalg.norm(xo)
