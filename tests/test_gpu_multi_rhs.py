"""The several-right-hand-side solve at the edges of its forms: one launch for
small systems (256 and 1024 threads, one and four rows a thread), staged
products with few and many components, rows too long for the stage, and a
solution written over its right-hand side."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

from pflotran_amd import abi, runtime

pytestmark = pytest.mark.gpu


def system(n, long_rows, seed):
    """Strictly dominant by rows (diagonal 4, off-diagonal sum below 2): the inverse's infinity norm is below 1/2."""
    rng = np.random.default_rng(seed)
    A = sp.diags([rng.uniform(-0.5, 0.5, n - 1), np.full(n, 4.0), rng.uniform(-0.5, 0.5, n - 1)], [-1, 0, 1]).tolil()
    for i in range(n):
        A[i, (i * 7 + 3) % n] += 0.25 if (i * 7 + 3) % n != i else 0.0
    A = A.tocsr()
    if long_rows:
        rows = np.repeat(rng.choice(n, 30, replace=False), 300)
        A = A + sp.csr_matrix((np.full(rows.size, 0.001), (rows, rng.integers(0, n, rows.size))), shape=(n, n))
    A.sort_indices()
    return A


@pytest.mark.parametrize("n,comps,long_rows,in_place", [
    (1, 3, False, False), (255, 2, False, False), (256, 5, False, True), (257, 5, False, False),
    (1024, 1, False, False), (1025, 4, False, True), (4096, 3, False, False), (4097, 3, False, False),
    (4097, 1, False, True), (5003, 15, False, False), (5003, 2, True, False), (9001, 32, False, True)])
def test_solve_multi_matches_direct(n, comps, long_rows, in_place):
    import torch
    A = system(n, long_rows, n + comps) if n > 1 else sp.csr_matrix(np.array([[4.0]]))
    rng = np.random.default_rng(n)
    B = rng.normal(size=(n, comps)) * 10.0 ** rng.uniform(-3, 3, size=comps)
    dev = lambda a, t: torch.as_tensor(np.ascontiguousarray(a), dtype=t, device="cuda")  # noqa: E731
    vals, b = dev(A.data, torch.float64), dev(B, torch.float64)
    h = runtime.Bsr(dev(A.indptr, torch.int32), dev(A.indices, torch.int32), 1)
    x = b if in_place else torch.full_like(b, float("nan"))
    st = abi.KrylovStats()
    o = abi.KrylovOpts(rtol=1e-13)
    rc = h.lib.pfx_bsr_solve_multi(h.handle, vals.data_ptr(), b.data_ptr(), x.data_ptr(), comps, C.byref(o),
                                   torch.cuda.current_stream().cuda_stream, 0, C.byref(st))
    assert rc == 0 and st.reason == abi.PFX_KSP_CONVERGED_RTOL
    ref = spla.splu(A.tocsc()).solve(B)
    # |x - ref|_inf <= |A^-1|_inf |r|_2, r below 1e-13 |b|_2 by the recurrence and 1e-14 |b|_2 of its rounding
    bound = 0.5 * 1.1e-13 * np.linalg.norm(B, axis=0) + 1e-14 * np.abs(ref).max(axis=0)
    assert (np.abs(x.cpu().numpy() - ref).max(axis=0) <= bound).all()
    h.close()


def test_zero_right_hand_sides_and_breakdown():
    """A zero right-hand side converges at the start with x = 0; a zero pivot fails and leaves x = 0, in both forms."""
    import torch
    for n in (300, 6000):
        A = system(n, False, 3)
        dev = lambda a, t: torch.as_tensor(np.ascontiguousarray(a), dtype=t, device="cuda")  # noqa: E731
        for pivot in (True, False):
            if not pivot:
                A[5, 5] = 0.0
            vals = dev(A.data, torch.float64)
            h = runtime.Bsr(dev(A.indptr, torch.int32), dev(A.indices, torch.int32), 1)
            b = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
            if not pivot:
                b += 1.0
            x = torch.full_like(b, 7.0)
            st = abi.KrylovStats()
            rc = h.lib.pfx_bsr_solve_multi(h.handle, vals.data_ptr(), b.data_ptr(), x.data_ptr(), 3, None,
                                           torch.cuda.current_stream().cuda_stream, 0, C.byref(st))
            assert rc == 0 and st.iterations == 0
            assert (st.reason > 0) == pivot and bool((x == 0).all())
            h.close()
