"""How the several-right-hand-side solve ends, on both sides of the 4096 rows up
to which it is one launch, waited for and enqueued: a column decided at the
start beside running ones, an iteration limit, a breakdown in the first
iteration, every column's breakdown; and grids and the operator-split graph
above 4096 rows."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import oracle as orc
from chemdefs import carbonate_column
from pflotran_amd import abi, column, runtime
from test_column_os import initial_state, react_opts
from test_gpu_multi_rhs import system
from test_gpu_os_transport import random_grid, rel_err

pytestmark = pytest.mark.gpu
SIZES = (300, 1500, 4096, 4097, 6001)


def solve(A, B, ordered, **opts):
    """x (pre-filled with 7) and the statistics."""
    import torch
    dev = lambda a, t: torch.as_tensor(np.ascontiguousarray(a), dtype=t, device="cuda")  # noqa: E731
    vals, b = dev(A.data, torch.float64), dev(B, torch.float64)
    h = runtime.Bsr(dev(A.indptr, torch.int32), dev(A.indices, torch.int32), 1)
    x, st, o = torch.full_like(b, 7.0), abi.KrylovStats(), abi.KrylovOpts(**opts)
    s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = h.lib.pfx_bsr_solve_multi(h.handle, vals.data_ptr(), b.data_ptr(), x.data_ptr(), B.shape[1], C.byref(o), s,
                                   ordered, C.byref(st))
    assert rc == 0
    if ordered:
        assert h.lib.pfx_bsr_multi_stats(h.handle, s, C.byref(st)) == 0
    x = x.cpu().numpy()
    h.close()
    return x, st


def bicgstab(A, b, its):
    """`its` iterations of BiCGStab from zero, right-preconditioned by the diagonal."""
    d = 1.0 / A.diagonal()
    x, r = np.zeros_like(b), b.copy()
    p = r.copy()
    rho = b @ r
    for _ in range(its):
        v = A @ (d * p)
        alpha = rho / (b @ v)
        s = r - alpha * v
        t = A @ (d * s)
        omega = (t @ s) / (t @ t)
        x += d * (alpha * p + omega * s)
        r = s - omega * t
        new = b @ r
        p = r + (new / rho) * (alpha / omega) * (p - omega * v)
        rho = new
    return x


@pytest.mark.parametrize("ordered", [0, 1])
@pytest.mark.parametrize("n", SIZES)
def test_zero_column_beside_running_ones(n, ordered):
    A = system(n, False, n)
    rng = np.random.default_rng(n)
    B = rng.normal(size=(n, 4))
    B[:, 1] = 0.0
    x, st = solve(A, B, ordered, rtol=1e-13, max_iterations=60)
    assert st.reason == abi.PFX_KSP_CONVERGED_ATOL          # the zero column's, the worst of them
    assert (x[:, 1] == 0.0).all()
    ref = spla.splu(A.tocsc()).solve(B)
    # as in test_gpu_multi_rhs: |A^-1|_inf below 1/2, the residual by recurrence and its rounding
    assert (np.abs(x - ref).max(axis=0) <= 0.5 * 1.1e-13 * np.linalg.norm(B, axis=0) + 1e-14 * np.abs(ref).max()).all()


@pytest.mark.parametrize("ordered", [0, 1])
@pytest.mark.parametrize("its", [1, 2, 5])
@pytest.mark.parametrize("n", SIZES)
def test_iteration_limit(n, its, ordered):
    """The iterate after `its` iterations against plain BiCGStab: dot products of n terms agree to n eps (1e-12), and
    each iteration passes their error on with a factor of a few (condition number below 3): 1e-9 of the largest."""
    A = system(n, False, n + 1)
    B = np.random.default_rng(n).normal(size=(n, 3))
    x, st = solve(A, B, ordered, rtol=1e-14, max_iterations=its)
    assert st.reason == abi.PFX_KSP_DIVERGED_ITS and st.iterations == 3 * its
    for c in range(3):
        ref = bicgstab(A, B[:, c].copy(), its)
        assert np.abs(x[:, c] - ref).max() <= 1e-9 * np.abs(ref).max()


def breaking(n):
    """Blocks [[1, -2], [0, 1]]: for b = (1, 1, ...) the sum (b, A b) of whole numbers is exactly zero."""
    n -= n % 2
    return sp.csr_matrix(sp.block_diag([np.array([[1.0, -2.0], [0.0, 1.0]])] * (n // 2))), n


@pytest.mark.parametrize("ordered", [0, 1])
@pytest.mark.parametrize("n", SIZES)
def test_first_iteration_breakdown(n, ordered):
    """The column that breaks down keeps its start, zero; the others (minimal polynomial of degree 2) are solved."""
    A, n = breaking(n)
    B = np.random.default_rng(n).normal(size=(n, 3))
    B[:, 1] = 1.0
    x, st = solve(A, B, ordered, rtol=1e-12, max_iterations=20)
    assert st.reason == abi.PFX_KSP_DIVERGED_BREAKDOWN
    assert (x[:, 1] == 0.0).all()
    ref = spla.splu(A.tocsc()).solve(B)
    for c in (0, 2):   # |A^-1|_inf = 3
        assert np.abs(x[:, c] - ref[:, c]).max() <= 3 * 1.1e-12 * np.linalg.norm(B[:, c])
    x, st = solve(A, B[:, 1:2], ordered, rtol=1e-12, max_iterations=20)
    assert st.reason == abi.PFX_KSP_DIVERGED_BREAKDOWN and st.iterations == 1 and (x == 0.0).all()


@pytest.mark.parametrize("shape,N", [((17, 16, 16), 4), ((33, 2, 64), 15), ((4100, 1, 1), 5), ((3, 41, 40), 32)])
def test_transport_above_one_launch(shape, N):
    """The transport step on grids above 4096 rows against the oracle's direct solve, to the bound of the small ones;
    enqueued, the same bits."""
    import torch
    rng = np.random.default_rng(sum(shape) + N)
    nx, ny, nz = shape
    n = nx * ny * nz
    f = random_grid(rng, nx, ny, nz, N)
    phi, vol = rng.uniform(0.1, 0.4, size=n), rng.uniform(0.5, 2.0, size=n)
    dt = 3600.0
    T = rng.uniform(1e-5, 1e-2, size=(n, N))
    ref = orc.os_transport_step(orc.HostGrid(nx, ny, nz, **f), phi * 1000.0 * vol / dt, T)
    g = runtime.DeviceGrid(nx, ny, nz, **f)
    dev = lambda a: torch.as_tensor(a, device="cuda").clone()  # noqa: E731
    outs = []
    for ordered in (0, 1):
        dc = runtime.DeviceCells({"total": dev(T), "porosity": dev(phi), "volume": dev(vol)}, n)
        tr = runtime.OsTransport(g)
        o = abi.default_opts(dt=dt, saturation=1.0)
        o.stream_ordered = ordered
        rc, st = tr.step(dc, g, N, o, rtol=1e-13, max_iterations=60)
        torch.cuda.synchronize()
        assert rc == 0 and (ordered or st.reason == abi.PFX_KSP_CONVERGED_RTOL)
        outs.append(dc.t["total"].cpu().numpy())
        tr.close()
    assert rel_err(outs[0], ref) <= 1e-10
    assert np.array_equal(outs[0], outs[1])


def test_step_graph_above_one_launch():
    """The captured operator-split step of a 4500-cell column: every replay, with the eager steps in between, leaves
    the eager step's bits."""
    import torch
    t = carbonate_column()
    col = column.Column(ncells=4500)
    cells, inflow = initial_state(t, col.ncells)
    dt = 86400.0
    tab = runtime.Tables(t)
    f = column.grid_faces(col, inflow)
    grid = runtime.DeviceGrid(f["nx"], f["ny"], f["nz"], f["q"], f["dd"], area=f["area"], bc_q=f["bc_q"],
                              bc_dd=f["bc_dd"], bc_total=f["bc_total"])
    o_t = abi.default_opts(dt=dt, porosity=col.porosity, saturation=col.saturation, volume=col.volume)
    de, dg = (runtime.DeviceCells.from_host(dict(cells.arrays), col.ncells) for _ in range(2))
    tr_e, tr_g = runtime.OsTransport(grid), runtime.OsTransport(grid)
    graph = runtime.OsStepGraph(tr_g, grid, tab, dg, t.N, o_t, react_opts(dt), rtol=1e-12, max_iterations=30)
    for step in range(4):
        rc, ts = tr_e.step(de, grid, t.N, o_t, rtol=1e-12, max_iterations=30)
        assert rc == 0
        rc, st = runtime.react_batch(tab, de, react_opts(dt))
        runtime.update_kinetic_state(tab, de, react_opts(dt))
        torch.cuda.synchronize()
        graph.launch()
        rc_g, st_g, ks_g = graph.stats()
        assert rc_g == rc and st_g.total_iterations == st.total_iterations
        assert ks_g.reason == ts.reason == abi.PFX_KSP_CONVERGED_RTOL and ks_g.iterations == ts.iterations
        for k in ("total", "pri_molal", "mnrl_volfrac", "pri_act_coef"):
            assert torch.equal(dg.t[k], de.t[k]), (step, k)
    graph.close()
    tr_e.close()
    tr_g.close()
