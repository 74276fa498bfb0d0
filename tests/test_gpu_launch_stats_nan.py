"""The largest scaled residual of a launch where some are not finite: NaN if any
cell's is, as a reduction over the per-cell values gives it."""
import numpy as np
import pytest

from pflotran_amd import abi, runtime, synth, workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,bad", [(1, [0]), (300, [299]), (5000, [0, 1700, 4999]), (70001, [65536])])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_residuals_that_are_not_finite(n, bad, value):
    t = synth.random_network(5, 8, 1, ionx=False)
    tab = runtime.Tables(t)
    dc, _ = workload.speciated_cells(t, tab, n)
    for i in bad:
        dc.t["total"][i, 1] = value
    rc, st = runtime.react_batch(tab, dc, synth.react_opts(guess_mode=abi.PFX_GUESS_PREVIOUS, max_iterations=20))
    out = dc.to_host()
    rr, status, it = out["rel_res"], out["status"], out["num_iterations"]
    assert (status[bad] != 0).all() and not np.isfinite(rr[bad]).all()
    assert rc == n - st.converged == np.count_nonzero(status)
    assert st.total_iterations == it.sum(dtype=np.int64)
    want = np.nan if np.isnan(rr).any() else np.abs(rr).max()
    assert st.max_rel_res == want or (np.isnan(want) and np.isnan(st.max_rel_res))
