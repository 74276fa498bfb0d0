"""Activity coefficients that a call does not form come back as they were
given, bit for bit: the aux-var refresh without an activity pass, in each group
width."""
import numpy as np
import pytest

from gpu_cases import host_arrays, speciated_state
from pflotran_amd import runtime, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [7, 15, 20])
def test_refresh_without_an_activity_pass_keeps_the_coefficients(N):
    t = synth.random_network(N, 2 * N, 2, ionx=True, seed=synth.SEED + N)
    cells, _, _, _ = speciated_state(t, 97)
    # coefficients of all sizes, so that a rounded copy of some would show
    rng = np.random.default_rng(N)
    cells["sec_act_coef"][:] = np.exp(rng.uniform(-3.0, 1.0, size=cells["sec_act_coef"].shape))
    cells["pri_act_coef"][:] = np.exp(rng.uniform(-1.0, 0.5, size=cells["pri_act_coef"].shape))
    dc = runtime.DeviceCells.from_host(host_arrays(cells), 97)
    tab = runtime.Tables(t)
    for _ in range(3):
        runtime.auxvar(tab, dc, 0, synth.react_opts())
    out = dc.to_host()
    assert np.array_equal(out["sec_act_coef"], cells["sec_act_coef"])
    assert np.array_equal(out["pri_act_coef"], cells["pri_act_coef"])
    # a pass that forms them does change them
    runtime.auxvar(tab, dc, 1, synth.react_opts())
    assert not np.array_equal(dc.to_host()["sec_act_coef"], cells["sec_act_coef"])
