"""sfa_system_apply on device vectors: bit for bit the oracle's product, straight
from the caller's vectors."""
import numpy as np
import pytest

import oracle
from simplefem_amd import capi
from simplefem_amd import systems as S
from simplefem_amd.hipmem import DeviceArray

pytestmark = pytest.mark.gpu


def _rows_of(widths, seed):
    """A matrix whose row i has widths[i] entries, in random column order."""
    rng = np.random.default_rng(seed)
    n = len(widths)
    A = np.concatenate([[0], np.cumsum(widths)]).astype(np.int32)
    C = np.concatenate([rng.permutation(n)[:w] for w in widths]).astype(np.int32)
    return S.CSRSystem("rows", n, A, C, rng.uniform(-1, 1, C.size), np.zeros(n, dtype=bool))


# empty rows, the 16 entries loaded ahead, the chunks of 8 after them, slices of
# one and of several widths, a last slice of one row
CASES = {
    "one": lambda: _rows_of([1], 1),
    "empty_rows": lambda: _rows_of([0, 3, 0, 0, 5, 1] * 30, 2),
    "w16": lambda: _rows_of([16] * 65, 3),
    "w17": lambda: _rows_of([17] * 64, 4),
    "w24_25": lambda: _rows_of([24, 25] * 80, 5),
    "uneven": lambda: _rows_of(list(range(0, 129)), 6),
    "kuhn_20": lambda: S.poisson3d_p1_kuhn(20),
}


@pytest.mark.parametrize("lanes", [1, 2, 4, 8])
@pytest.mark.parametrize("name", sorted(CASES))
def test_apply_on_device_vectors(name, lanes):
    s = CASES[name]()
    src = S.uniform_pm1(3, s.n)
    src[0] = np.inf  # only rows that read it may see it (padding entries do not)
    want = oracle.csr_apply(s.n, s.A, s.C, s.V, src, 1.75)
    with capi.System(capi.METHOD_CG, s.n, s.A, s.C, s.V) as system:
        system.set_spmv(lanes)
        x, y = DeviceArray.from_host(src), DeviceArray(s.n)
        system.apply(y, x, 1.75)
        assert np.array_equal(y.download(), want, equal_nan=True)
        host = np.empty(s.n)
        system.apply(host, src, 1.75)
        assert np.array_equal(host, want, equal_nan=True)
        system.apply(x, x, 1.75)  # in place
        assert np.array_equal(x.download(), want, equal_nan=True)
