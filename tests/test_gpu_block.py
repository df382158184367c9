"""Small systems run in one workgroup (csrc/block_solve.hpp): batch slots whose
two gathered vectors fit a CU's LDS.

The bars are those of the batch engine: K within max(1, 2%) of the oracle's,
the same exit reason, x within 1e-10 relative; and a run cut into pieces gives
the bits of one run.
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
