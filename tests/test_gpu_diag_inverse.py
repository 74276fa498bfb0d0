"""The inverted diagonal blocks of the block solver: on a matrix without
couplings the preconditioned operator is the identity, so the solve ends
after one iteration (up to rounding: three are allowed) on the blocks' own
solutions.  The blocks are Gaussian, so that every step has to look for its
pivot; a few are permutations, with exact zeros at every position but one."""
import numpy as np
import pytest

from pflotran_amd import abi, runtime
from test_gpu_gi_solver import faces

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 2, 7, 8, 9, 15, 16, 17, 24, 31, 32])
def test_inverted_blocks(N):
    """The residual to 1e-11 of ||b|| (the solve's 1e-12 and the rounding of one product); a solution's
    distance from numpy's to that residual times the largest ||A^-1||."""
    import torch
    rng = np.random.default_rng(100 + N)
    g = runtime.DeviceGrid(5, 4, 3, *faces(rng, 5, 4, 3))
    rp, ci = runtime.gi_structure(g)
    rp_h, ci_h = rp.cpu().numpy(), ci.cpu().numpy()
    n = len(rp_h) - 1
    A = rng.normal(size=(n, N, N))
    A[::7] = [np.eye(N)[rng.permutation(N)] * 3.0 for _ in A[::7]]
    vals = np.zeros((len(ci_h), N, N))
    for row in range(n):
        b = rp_h[row] + int(np.flatnonzero(ci_h[rp_h[row]:rp_h[row + 1]] == row)[0])
        vals[b] = A[row].T                                   # column-major blocks
    b = rng.normal(size=(n, N))
    bsr = runtime.Bsr(rp, ci, N)
    x, st = bsr.solve(torch.as_tensor(vals, device="cuda"), torch.as_tensor(b, device="cuda"), rtol=1e-12)
    bsr.close()
    x = x.cpu().numpy()
    assert st.reason == abi.PFX_KSP_CONVERGED_RTOL and st.iterations <= 3
    assert np.linalg.norm(np.einsum("nij,nj->ni", A, x) - b) <= 1e-11 * np.linalg.norm(b)
    ref = np.linalg.solve(A, b[..., None])[..., 0]
    inv = np.linalg.norm(np.linalg.inv(A), 2, axis=(1, 2)).max()
    assert np.linalg.norm(x - ref) <= 1e-11 * inv * np.linalg.norm(b)
