"""Solves of middle-sized systems in one launch of a team of workgroups
(csrc/team.hip).

Its rows and sums are those of the launches of an iteration, which
sfa_system_profile runs: x, residual, K and z.r agree bit for bit, whichever
of the two a solve takes and wherever it changes over.
"""
import ctypes
import threading

import numpy as np
import pytest

import oracle
from simplefem_amd import capi
from simplefem_amd import systems as S
from simplefem_amd.hipmem import check, hip

pytestmark = pytest.mark.gpu


def _shuffled(s, seed):
    """s with its unknowns renumbered at random: deep dependency levels in natural order."""
    return S.permute_symmetric(s, np.random.default_rng(seed).permutation(s.n), s.name + "_shuffled")


# just above the one-workgroup limit of 8,190 rows and larger; rows of up to
# 4, 8 and many entries a triangle; K above 256, the iterations of one launch;
# colours of few and many slices; natural order, where a row's two steps fall
# to different wavefronts, with 13 and with some hundred levels
CASES = {
    "p1_2d_91": (lambda: S.lagrange_pr(2, 90, 1), "rainbow"),
    "kuhn_21": (lambda: S.poisson3d_p1_kuhn(21), "rainbow"),
    "p3_2d_103": (lambda: S.lagrange_pr(2, 34, 3), "rainbow"),
    "p3_3d_22": (lambda: S.lagrange_pr(3, 7, 3), "rainbow"),
    "p2_2d_201": (lambda: S.lagrange_pr(2, 100, 2), "rainbow"),
    "hcurl_12": (lambda: S.hcurl3d_whitney_kuhn(12), "rainbow"),
    "reference_129": (lambda: S.poisson2d_p1(7, numbering="reference"), "ssor"),
    "axes_95": (lambda: S.lagrange_pr(2, 94, 1), "ssor"),
    "shuffled_95": (lambda: _shuffled(S.lagrange_pr(2, 94, 1), 3), "ssor"),
}


def _system(s, variant, **more):
    col = oracle.rainbow(s.n, s.A, s.C) if variant == "rainbow" else (0, None, None, None)
    method = capi.METHOD_RAINBOW if variant == "rainbow" else capi.METHOD_SSOR
    return capi.System(method, s.n, s.A, s.C, s.V, s.diagonal(), 1.2, *col, **more), col


def _solve(system, s, b):
    x, r, info = np.zeros(s.n), np.zeros(s.n), {}
    system.solve(x, b, r, 1e-10, info=info)
    return x, r, info


def _same(got, want):
    assert got[2]["iterations"] == want[2]["iterations"] and got[2]["zr"] == want[2]["zr"]
    assert got[2]["exit_reason"] == want[2]["exit_reason"]
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("name", sorted(CASES))
def test_team_is_bit_identical_to_launches(name):
    make, variant = CASES[name]
    s = make()
    b = S.rhs_uniform(s, 31)
    system, col = _system(s, variant)
    print(f"case: {name} {variant} n={s.n} nnz={s.nnz}", flush=True)
    with system:
        team = _solve(system, s, b)
        again = _solve(system, s, b)
        x, r = np.zeros(s.n), np.zeros(s.n)
        _, info = system.profile(x, b, r, 1e-10)
    _same(again, team)
    _same(team, (x, r, info))
    xo, _, io = oracle.solve(variant, s.A, s.C, s.V, b, aux=s.diagonal(), omega=1.2,
                             colouring=col if variant == "rainbow" else None)
    slack, bar = (0.04, 5e-9) if name.startswith("hcurl") else (0.02, 1e-10)
    assert abs(info["iterations"] - io["iterations"]) <= max(1, int(slack * io["iterations"]))
    assert np.abs(x - xo).max() <= bar * np.abs(xo).max()


def test_team_breakdown_on_nan():
    """A NaN right-hand side ends in breakdown (its NaN is not taken for a row
    that is not done)."""
    s = S.lagrange_pr(2, 94, 1)
    b = S.rhs_uniform(s, 3)
    b[s.n // 2] = np.nan
    for variant in ("rainbow", "ssor"):
        system, _ = _system(s, variant)
        with system:
            _, _, info = _solve(system, s, b)
        assert info["exit_reason"] == capi.EXIT_BREAKDOWN


def test_threads_change_over_between_team_and_launches():
    """A team runs only while its solve is alone: solves of four threads that
    overlap take the launches for part of their way, with the same bits."""
    s = S.hcurl3d_whitney_kuhn(12)
    bs = [S.rhs_uniform(s, 50 + k) for k in range(4)]
    systems = [_system(s, "rainbow", fp32_inner=True)[0] for _ in bs]
    alone = [_solve(system, s, b) for system, b in zip(systems, bs)]
    mixed = []
    for system, b in zip(systems, bs):
        x = np.zeros(s.n)
        mixed.append((x, system.solve_mixed(x, b, 1e-10)))
    got = [[] for _ in bs]

    def work(k):
        for _ in range(3):
            got[k].append(_solve(systems[k], s, bs[k]))
        x = np.zeros(s.n)
        got[k].append((x, systems[k].solve_mixed(x, bs[k], 1e-10)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for k in range(4):
        for solved in got[k][:-1]:
            _same(solved, alone[k])
        assert got[k][-1][1] == mixed[k][1] and np.array_equal(got[k][-1][0], mixed[k][0])
    for system in systems:
        system.close()


def test_team_without_room_gives_up():
    """On a stream that may use 32 CUs the team's workgroups are never all
    resident: its waits run out (50 ms) and the solve is made again by
    launches, to the same bits; later solves go there at once."""
    s = S.lagrange_pr(2, 94, 1)
    b = S.rhs_uniform(s, 8)
    system, _ = _system(s, "rainbow")
    lib = hip()
    lib.hipExtStreamCreateWithCUMask.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_uint32,
                                                 ctypes.POINTER(ctypes.c_uint32)]
    lib.hipStreamDestroy.argtypes = [ctypes.c_void_p]
    stream = ctypes.c_void_p()
    mask = (ctypes.c_uint32 * 8)(0xFFFFFFFF, *([0] * 7))
    check(lib.hipExtStreamCreateWithCUMask(ctypes.byref(stream), 8, mask))
    with system:
        want = _solve(system, s, b)
        system.set_stream(stream.value)
        for _ in range(2):
            _same(_solve(system, s, b), want)
        system.set_stream(None)
        _same(_solve(system, s, b), want)
    check(lib.hipStreamDestroy(stream))
