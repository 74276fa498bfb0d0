"""The unpivoted group solve at the edges of its group sizes: 8, 16 and 32
lanes per cell, the smallest and largest systems of each, and groups wider
than the system needs."""
from dataclasses import replace

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [(5, 0), (7, 0), (8, 0), (5, 16), (9, 0), (15, 0), (16, 0), (9, 32), (17, 0), (24, 0), (31, 0), (32, 0)]


@pytest.mark.parametrize("N,lanes", CASES)
def test_reaction_step_group_sizes(N, lanes):
    """Free ions to 1e-10 of the oracle, the parity bound of the reaction
    step, on the cells that FP64 resolves to 1e-11 (conditioning_floor; the
    step test stops below 1e-11), and every cell's status; an odd number of
    cells."""
    import oracle as orc
    from gpu_cases import conditioning_floor
    from pflotran_amd import abi, runtime, synth

    t = replace(synth.random_network(N, 2 * N, 2, ionx=True, seed=synth.SEED + N), group_lanes=lanes, _desc=None)
    n = 131
    cells, _, _, _ = orc.speciated_state(t, n)
    ref = cells.copy()
    opts = dict(guess_mode=abi.PFX_GUESS_PREVIOUS, max_iterations=300)
    orc.react_batch(t, ref, synth.react_opts(**opts))
    dc = runtime.DeviceCells.from_host({k: (None if v is None else v.copy()) for k, v in cells.arrays.items()}, n)
    runtime.react_batch(runtime.Tables(t), dc, synth.react_opts(**opts))
    out = dc.to_host()
    both = (out["status"] == 0) & (ref["status"] == 0)
    assert both.mean() > 0.9 and np.array_equal(out["status"], ref["status"])
    both &= conditioning_floor(t, ref, cells, synth.STEP_DT) <= 1e-11
    assert both.sum() > 40
    rel = np.abs(out["pri_molal"][both] - ref["pri_molal"][both]) / ref["pri_molal"][both]
    assert rel.max() <= 1e-10
