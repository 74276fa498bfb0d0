"""A launch's statistics against the per-cell outputs they are formed from:
batches around a wavefront, a workgroup, the cells of one workgroup and more than
the workgroups' one pass.  Whole numbers and a maximum, so exactly equal."""
import numpy as np
import pytest

from pflotran_amd import abi, runtime, synth, workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 65, 255, 257, 1024, 1025, 65537, 262145])
@pytest.mark.parametrize("iterations", [2, 100])
def test_statistics(n, iterations):
    """Cells of unlike length, some of which two iterations do not finish; a step of n speciated cells."""
    t = synth.random_network(5, 8, 1, ionx=False)
    tab = runtime.Tables(t)
    dc, _ = workload.speciated_cells(t, tab, n)
    rc, st = runtime.react_batch(tab, dc, synth.react_opts(guess_mode=abi.PFX_GUESS_DEFAULT, max_iterations=iterations))
    out = dc.to_host()
    it, status, rr = out["num_iterations"], out["status"], out["rel_res"]
    assert st.ncells == n and st.converged == np.count_nonzero(status == 0) and rc == n - st.converged
    assert st.total_iterations == it.sum(dtype=np.int64)
    assert st.max_iterations == it.max() and st.min_iterations == it.min()
    hist = np.bincount(np.minimum(it, 31), minlength=32)
    assert list(st.iteration_histogram) == list(hist)
    if np.isfinite(rr).all():
        assert st.max_rel_res == np.abs(rr).max()
