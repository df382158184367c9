"""Systems of so many rows that the search direction is stored by a kernel of its
own, ahead of the product: the last size with one kernel, the first with two, and
a size whose product takes two rounds, with empty rows among the others.  The
residual recomputed from x bounds the error; tolerances follow from that."""
import numpy as np
import pytest
import scipy.sparse as sp

import oracle
from simplefem_amd import capi
from simplefem_amd import systems as S

pytestmark = pytest.mark.gpu

ONE = 4 * 1024 * 64   # most rows of one kernel
ROUND = 4 * 2048 * 64  # most rows of one round of the product


def _band(n):
    """4 on the diagonal, -1 at distance 1, -1/2 at distance 7, and every 101st
    row and column empty: symmetric, with a spectrum in [1, 7] off the empty rows."""
    M = sp.diags_array([-0.5, -1.0, 4.0, -1.0, -0.5], offsets=[-7, -1, 0, 1, 7], shape=(n, n))
    keep = (np.arange(n) % 101 != 0).astype(float)
    M = (sp.diags_array(keep) @ M @ sp.diags_array(keep)).tocsr()
    M.eliminate_zeros()
    M.sort_indices()
    return S.CSRSystem("band", n, M.indptr.astype(np.int32), M.indices.astype(np.int32), M.data, keep == 0)


@pytest.mark.parametrize("method", ["cg", "jacobi", "rainbow"])
@pytest.mark.parametrize("n", [ONE, ONE + 1, ROUND + 65])
def test_solutions_at_the_edges(n, method):
    s = _band(n)
    b = S.rhs_uniform(s, 4)
    diag = np.where(s.dirichlet, 0.0, 4.0)
    kind = {"cg": capi.METHOD_CG, "jacobi": capi.METHOD_DIAGONAL, "rainbow": capi.METHOD_RAINBOW}[method]
    aux = {"cg": None, "jacobi": np.full(n, 0.25), "rainbow": diag}[method]
    colours = oracle.rainbow(n, s.A, s.C) if method == "rainbow" else (0, None, None, None)
    x, r, info = np.zeros(n), np.zeros(n), {}
    with capi.System(kind, n, s.A, s.C, s.V, aux, 1.0, *colours, fp32_inner=True) as system:
        K = system.solve(x, b, r, 1e-10, info=info)
        assert system.stats()["kernels_per_iteration"] >= 2 + (n > ONE)
        # the least eigenvalue is 1 or more: |x - x*| <= |b - A x|
        res = b - oracle.csr_apply(n, s.A, s.C, s.V, x)
        assert 3 < K < 200
        assert np.linalg.norm(res) <= 2e-10 * np.linalg.norm(b)
        assert np.abs(res - r).max() <= 64 * K * np.finfo(float).eps * np.abs(b).max()
        # and with one kernel for both (two lanes per row): the same sums in
        # another order, so the iterates agree to what a run of K steps loses
        y = np.zeros(n)
        system.set_spmv(2)
        assert abs(system.solve(y, b, r, 1e-10) - K) <= 1
        assert np.abs(x - y).max() <= 4e-10 * np.linalg.norm(b)
        z = np.zeros(n)
        system.set_spmv(1)
        assert system.solve_mixed(z, b, 1e-10)["success"]
        assert np.linalg.norm(b - oracle.csr_apply(n, s.A, s.C, s.V, z)) <= 2e-10 * np.linalg.norm(b)
