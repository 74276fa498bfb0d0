"""One evaluation on a grid as a call: its launches' times are read, and it
costs the host one wait, as an evaluation without a grid does."""
import ctypes as C

import numpy as np
import pytest

from pflotran_amd import runtime, synth, workload
from test_gpu_call_costs import least
from test_gpu_gi import faces

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1), (5, 4, 1), (20, 18, 16)])
def test_times_and_cost(shape):
    """The times of both launches, within the call's; the call beside its launches no more than 1.4 times the plain
    evaluation's (1.5 to 1.8 with a wait between the launches)."""
    import torch
    nx, ny, nz = shape
    n = nx * ny * nz
    t = synth.random_network(8, 16, 2, ionx=False)
    tab = runtime.Tables(t)
    dc, _ = workload.speciated_cells(t, tab, n, oversample=2.0)
    q, dd = faces(np.random.default_rng(1), nx, ny, nz)
    grid = runtime.DeviceGrid(nx, ny, nz, q, dd, log_formulation=True)
    rp, _ = runtime.gi_structure(grid)
    dev = lambda *s: torch.empty(s, dtype=torch.float64, device="cuda")  # noqa: E731
    res, vals, jac = dev(n, 8), dev(int(rp[-1]), 8, 8), dev(n, 8, 8)
    o, cs, g = synth.react_opts(), dc.struct(), grid.struct()
    o.stream = torch.cuda.current_stream().cuda_stream
    lib = tab.lib if hasattr(tab, "lib") else runtime.load_library()

    def on_grid():
        assert lib.pfx_gi_residual_jacobian(tab.handle, C.byref(cs), C.byref(g), C.byref(o), rp.data_ptr(),
                                            res.data_ptr(), vals.data_ptr()) == 0

    def plain():
        assert lib.pfx_residual_jacobian(tab.handle, C.byref(cs), C.byref(o), res.data_ptr(), jac.data_ptr()) == 0
    t_grid = least(on_grid, 60)
    cell, flux = tab.timing()
    assert cell > 0.0 and flux > 0.0 and (cell + flux) * 1e-3 < 2.0 * t_grid
    t_plain = least(plain, 60)
    ev, none = tab.timing()
    assert ev > 0.0 and none == 0.0
    assert t_grid - (cell + flux) * 1e-3 <= 1.4 * (t_plain - ev * 1e-3)
