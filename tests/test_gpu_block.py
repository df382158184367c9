"""Small systems run in one workgroup (csrc/block_solve.hpp): Systems and batch
slots whose two gathered vectors fit a CU's LDS.

The bars are those of the solvers: K within max(1, 2%) of the oracle's, the
same exit reason, x within 1e-10 relative; and a run cut into pieces gives the
bits of one run.
"""
import numpy as np
import pytest

import oracle
from simplefem_amd import capi
from simplefem_amd import systems as S

pytestmark = pytest.mark.gpu


def _diagonal_system(n):
    d = np.linspace(1.0, 3.0, n)
    return S.CSRSystem("diag", n, np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32),
                       d, np.zeros(n, dtype=bool))


def _inactive_system(n):
    """Every row a zero row: nothing to solve."""
    return S.CSRSystem("inactive", n, np.zeros(n + 1, dtype=np.int32), np.zeros(0, dtype=np.int32),
                       np.zeros(0), np.ones(n, dtype=bool))


# rows of 1 to 60 entries (none, one, two and many chunks of four), one slice
# and its remainders, one colour and dozens, and the largest sizes: the LDS
# offsets of n + 2 FP64 entries fill 16 bits at 8,190 rows, so 8,100 runs in
# one workgroup and 8,281 in the lockstep engine
CASES = {
    "one_row": lambda: _diagonal_system(1),
    "diag_65": lambda: _diagonal_system(65),
    "inactive_3": lambda: _inactive_system(3),
    "fd2d_8": lambda: S.fd_laplacian_2d(8),
    "spd_63": lambda: S.random_spd(63, 0.08, 4),
    "spd_129_wide": lambda: S.random_spd(129, 0.4, 5),
    "kuhn_9": lambda: S.poisson3d_p1_kuhn(9),
    "p3_3d_4": lambda: S.lagrange_pr(3, 4, 3),
    "hcurl_5": lambda: S.hcurl3d_whitney_kuhn(5),
    "p1_2d_90": lambda: S.lagrange_pr(2, 89, 1),
    "p1_2d_91": lambda: S.lagrange_pr(2, 90, 1),
}


def _add(batch, s, omega=1.0):
    col = oracle.rainbow(s.n, s.A, s.C)
    return batch.add_matrix(s.n, s.A, s.C, s.V, s.diagonal(), omega, *col), col


def _check(s, b, col, x, info, omega=1.0):
    xo, _, io = oracle.solve("rainbow", s.A, s.C, s.V, b, aux=s.diagonal(), omega=omega, colouring=col)
    assert abs(info["iterations"] - io["iterations"]) <= max(1, int(0.02 * io["iterations"])), (s.name, info, io)
    assert info["exit_reason"] == io["exit_reason"], (s.name, info, io)
    assert np.abs(x - xo).max() <= 1e-10 * max(np.abs(xo).max(), 1e-300), s.name


@pytest.mark.parametrize("name", sorted(CASES))
def test_batch_slot_matches_oracle(name):
    s = CASES[name]()
    print(f"case: {name} n={s.n} nnz={s.nnz}", flush=True)
    with capi.Batch(max_slots=4) as batch:
        mid, col = _add(batch, s, 1.2)
        bs = [S.rhs_uniform(s, 60 + k) for k in range(3)]
        slots = batch.submit_group(mid, bs)
        while batch.run(0) > 0:
            pass
        for slot, b in zip(slots, bs):
            x, info = batch.collect(slot, s.n)
            _check(s, b, col, x, info, 1.2)


@pytest.mark.parametrize("mixed", [False, True])
def test_cut_runs_match_one_run(mixed):
    """Runs of 32 phases (one or two iterations at a time, restarts apart from
    iterations, mixed solves between corrections) against one run."""
    s = S.lagrange_pr(2, 7, 3)
    bs = [S.rhs_uniform(s, 80 + k) for k in range(2)]
    got = []
    for steps in (32, 0):
        with capi.Batch(mixed=mixed, max_slots=4) as batch:
            mid, _ = _add(batch, s)
            slots = [batch.submit(mid, b) for b in bs]
            calls = 0
            while batch.run(steps) > 0:
                calls += 1
            assert calls > 3 or steps == 0
            got.append([batch.collect(k, s.n) for k in slots])
    for (xa, ia), (xb, ib) in zip(*got):
        assert ia == ib
        assert np.array_equal(xa, xb)


def test_batch_slot_breakdown_and_nan():
    """A NaN right-hand side ends in breakdown alone, beside a good one."""
    s = S.poisson2d_p1(4)
    good, bad = S.rhs_uniform(s, 1), S.rhs_uniform(s, 2)
    bad[s.n // 2] = np.nan
    with capi.Batch(max_slots=4) as batch:
        mid, col = _add(batch, s)
        slots = batch.submit_group(mid, [bad, good])
        while batch.run(0) > 0:
            pass
        _, info = batch.collect(slots[0], s.n)
        assert info["exit_reason"] == capi.EXIT_BREAKDOWN and not info["success"]
        x, info = batch.collect(slots[1], s.n)
        _check(s, good, col, x, info)


METHODS = {"cg": capi.METHOD_CG, "jacobi": capi.METHOD_DIAGONAL, "ssor": capi.METHOD_SSOR,
           "rainbow": capi.METHOD_RAINBOW}


def _solve(variant, s, b, x0=None, r0=None, omega=1.2, precision=1e-10):
    """(system's, oracle's) x, residual and info of one solve."""
    col = oracle.rainbow(s.n, s.A, s.C) if variant == "rainbow" else (0, None, None, None)
    d = s.diagonal()
    aux = {"cg": None, "jacobi": np.divide(1.0, d, out=np.zeros(s.n), where=d != 0)}.get(variant, d)
    x = np.zeros(s.n) if x0 is None else x0.copy()
    r = np.zeros(s.n) if r0 is None else r0.copy()
    info = {}
    with capi.System(METHODS[variant], s.n, s.A, s.C, s.V, aux, omega, *col) as system:
        system.solve(x, b, r, precision, info=info)
    want = oracle.solve(variant, s.A, s.C, s.V, b, x0=x0, residual0=r0, precision=precision,
                        aux=aux, omega=omega, colouring=col if variant == "rainbow" else None)
    return (x, r, info), want


@pytest.mark.parametrize("variant", sorted(METHODS))
@pytest.mark.parametrize("name", sorted(CASES))
def test_system_matches_oracle(name, variant):
    """Nonzero x0 and residual0: rows a variant skips keep theirs."""
    s = CASES[name]()
    rng = np.random.default_rng(5)
    b, x0, r0 = (rng.uniform(-1, 1, s.n) for _ in range(3))
    b[s.diagonal() == 0] = 0.0
    print(f"case: {variant} {name} n={s.n} nnz={s.nnz}", flush=True)
    (x, r, info), (xo, ro, io) = _solve(variant, s, b, x0, r0)
    assert abs(info["iterations"] - io["iterations"]) <= max(1, int(0.02 * io["iterations"])), (info, io)
    assert info["exit_reason"] == io["exit_reason"], (info, io)
    bad = np.isnan(xo)
    assert np.array_equal(np.isnan(x), bad) and np.array_equal(np.isnan(r), np.isnan(ro))
    if bad.any():
        return
    assert np.abs(x - xo).max() <= 1e-10 * max(np.abs(xo).max(), 1e-300)
    # The loop may end an iteration earlier or later than the oracle's, so the
    # residual is held against its own x: the recurrence drifts from b - A x by
    # rounding only, a few hundred units in the last place of |A||x|.
    true = b - oracle.csr_apply(s.n, s.A, s.C, s.V, x)
    size = oracle.csr_apply(s.n, s.A, s.C, np.abs(s.V), np.abs(x)) + np.abs(b)
    kept = (s.diagonal() == 0) & (variant != "cg")
    assert np.array_equal(r[kept], r0[kept]) and np.array_equal(x[kept], x0[kept])
    assert np.abs(r - true)[~kept].max(initial=0.0) <= 1e-13 * max(size.max(initial=0.0), 1e-300)


def test_many_iterations_take_several_launches():
    """One launch runs at most 4,096 iterations.  CG on the 1D Laplacian of
    8,000 rows needs about as many as there are rows; its condition number is
    2.6e7, so two FP64 solves agree to some 1e-8 and no better."""
    n = 8000
    rows = np.repeat(np.arange(n), 3)
    cols = rows + np.tile([-1, 0, 1], n)
    vals = np.tile([-1.0, 2.0, -1.0], n)
    keep = (cols >= 0) & (cols < n)
    A = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=n))]).astype(np.int32)
    s = S.CSRSystem("laplace1d", n, A, cols[keep].astype(np.int32), vals[keep], np.zeros(n, dtype=bool))
    b = S.uniform_pm1(7, n)
    (x, _, info), (xo, _, io) = _solve("cg", s, b, precision=1e-9)
    print(f"case: 1D Laplacian, K {info['iterations']} oracle {io['iterations']}", flush=True)
    assert io["iterations"] > 4096
    assert info["exit_reason"] == io["exit_reason"]
    assert abs(info["iterations"] - io["iterations"]) <= 0.02 * io["iterations"]
    assert np.linalg.norm(x - xo) <= 1e-7 * np.linalg.norm(xo)


def test_mixed_solve_continues_directions():
    """The FP32 inner solves in one workgroup: the FP64 residual target is met,
    and inner solves continue the previous one's direction."""
    s = S.poisson3d_p1_kuhn(16)
    b = S.rhs_uniform(s, 9)
    col = oracle.rainbow(s.n, s.A, s.C)
    with capi.System(capi.METHOD_RAINBOW, s.n, s.A, s.C, s.V, s.diagonal(), 1.0, *col,
                     fp32_inner=True) as system:
        x = np.zeros(s.n)
        info = system.solve_mixed(x, b, 1e-10, inner_rtol=1e-2)
    res = b - oracle.csr_apply(s.n, s.A, s.C, s.V, x)
    res[s.dirichlet] = 0.0
    assert info["success"] and np.linalg.norm(res) <= 1.0000001e-10 * np.linalg.norm(b)
    assert info["outer"] >= 3 and 1 <= info["continued"] < info["outer"]
