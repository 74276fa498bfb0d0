"""The grid evaluation's blocks over the sizes that its writes distinguish:
8-, 16- and 32-lane groups with full and partial rows, grids one cell thick in
each direction, and a network so large that the workgroup is halved."""
import numpy as np
import pytest

import oracle as orc
from gpu_cases import host_arrays, speciated_state
from pflotran_amd import runtime, synth
from test_gpu_gi import faces

pytestmark = pytest.mark.gpu


def check(t, shape, tab=None):
    """Residual to 1e-12 of its cell's accumulation, blocks to 2e-12 of their row's largest entry: the bounds of the
    15-component parity test."""
    nx, ny, nz = shape
    n = nx * ny * nz
    rng = np.random.default_rng(n + t.N)
    q, dd = faces(rng, nx, ny, nz)
    bc = dict(bc_q=(rng.normal(0, 1e-6, size=(nz, ny)), rng.normal(0, 1e-6, size=(nz, ny))),
              bc_dd=(np.full((nz, ny), 2e-7), np.full((nz, ny), 3e-7)), bc_total=(np.full(t.N, 1e-3), None))
    hg = orc.HostGrid(nx, ny, nz, q, dd, area=(0.5, 0.7, 0.9), log_formulation=True, **bc)
    cells, _, _, _ = speciated_state(t, n, seed=17)
    cells["pri_molal"][:] *= np.exp(0.2 * np.sin(np.arange(n * t.N)).reshape(n, t.N))
    r_o, v_o, rp_o, _ = orc.gi_residual_jacobian(t, cells, hg, synth.react_opts())
    dc = runtime.DeviceCells.from_host(host_arrays(cells), n)
    dg = runtime.DeviceGrid(nx, ny, nz, q, dd, area=(0.5, 0.7, 0.9), log_formulation=True, **bc)
    rp, _ = runtime.gi_structure(dg)
    r_g, v_g = runtime.gi_residual_jacobian(tab or runtime.Tables(t), dc, dg, synth.react_opts(), rp)
    r_g, v_g = r_g.cpu().numpy(), v_g.transpose(1, 2).cpu().numpy()
    acc = 0.25 * 1000.0 * np.abs(cells["total"]) / synth.STEP_DT
    assert np.max(np.abs(r_g - r_o) / (acc + np.abs(r_o) + 1e-300)) <= 1e-12
    for row in range(n):
        b = slice(rp_o[row], rp_o[row + 1])
        rowmax = np.abs(v_o[b]).max(axis=(0, 2))
        assert np.max(np.abs(v_g[b] - v_o[b]) / rowmax[None, :, None]) <= 2e-12, row


@pytest.mark.parametrize("N", [5, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 1, 3), (1, 5, 1), (4, 3, 5)])
def test_blocks(N, shape):
    check(synth.random_network(N, 2 * N, 2, ionx=False, seed=synth.SEED + N), shape)


def test_blocks_of_the_largest_network():
    for M in range(240, 60, -4):
        t = synth.random_network(16, M, 3, ionx=False, seed=synth.SEED + 5)
        try:
            tab = runtime.Tables(t)
        except runtime.PfxError:
            continue
        break
    check(t, (4, 3, 3), tab)
