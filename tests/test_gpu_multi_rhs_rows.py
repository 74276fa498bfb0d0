"""The several-right-hand-side solve at the number of matrix entries up to which
a small system is one launch, and with the launches' kernels on few rows of many
entries."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from pflotran_amd import abi
from test_gpu_call_costs import solve_time
from test_gpu_multi_rhs_ends import solve

pytestmark = pytest.mark.gpu


def rows_of(n, entries, seed):
    """n rows, `entries` in all, every row with its diagonal 3 and others that sum below 1: the inverse's infinity
    norm is below 1/2."""
    rng = np.random.default_rng(seed)
    count = entries // n + (np.arange(n) < entries % n)
    row = np.repeat(np.arange(n), count)
    j = np.arange(entries) - np.repeat(np.cumsum(count) - count, count)      # 0: the diagonal
    col = np.where(j == 0, row, (row + 1 + (j * 7919) % (n - 1)) % n)        # distinct: 7919 is no factor of n - 1
    val = np.where(j == 0, 3.0, rng.uniform(-1, 1, entries) / np.maximum(count, 2)[row])
    A = sp.csr_matrix((val, (row, col)), shape=(n, n))
    A.sort_indices()
    assert A.nnz == entries
    return A


@pytest.mark.parametrize("ordered", [0, 1])
@pytest.mark.parametrize("n,entries", [(250, 250 * 250), (300, 18000), (1000, 53248), (1000, 53249), (4096, 53248),
                                       (4096, 53249)])
@pytest.mark.parametrize("comps", [1, 3, 32])
def test_entries(n, entries, comps, ordered):
    A = rows_of(n, entries, n + entries)
    B = np.random.default_rng(n).normal(size=(n, comps))
    x, st = solve(A, B, ordered, rtol=1e-13, max_iterations=60)
    assert st.reason == abi.PFX_KSP_CONVERGED_RTOL
    ref = spla.splu(A.tocsc()).solve(B)
    # as in test_gpu_multi_rhs: the residual by recurrence and its rounding, through the inverse
    bound = 0.5 * 1.1e-13 * np.linalg.norm(B, axis=0) + 1e-14 * np.abs(ref).max()
    assert (np.abs(x - ref).max(axis=0) <= bound).all()


def test_long_rows_cost_no_more_below_the_limit_of_rows():
    """4000 rows of 200 entries took 6 times as long as 4200."""
    assert solve_time(4000, 200, 5) <= 2.0 * solve_time(4200, 200, 5)
