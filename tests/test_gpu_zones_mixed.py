"""Zoned launches that mix networks with and without mineral rate prefactors:
the kernel lays every zone's cells out with the prefactors' scalars, so the
launch has to be sized for that layout even where the largest zone has none.
The complexes are varied so that the sizes fall anywhere in the pieces by which
LDS is handed out."""
import numpy as np
import pytest

import oracle as orc
from gpu_cases import conditioning_floor, host_arrays, speciated_state
from pflotran_amd import abi, runtime, synth
from test_gpu_parity import _with_prefactors

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def prefactors():
    t = _with_prefactors(synth.random_network(15, 50, 3, ionx=True))
    return t, speciated_state(t, 61, seed=7)[0]


@pytest.mark.parametrize("N,M", [(8, M) for M in range(58, 66)] + [(15, 90), (15, 91), (15, 92), (30, 80), (30, 81)])
def test_mixed_zones_equal_separate_batches(prefactors, N, M):
    """Statuses equal, and free ions to 1e-10 (the step's parity bound) on the cells that FP64 resolves to 1e-11: the
    zone's network runs in another instantiation than its own batch.  Mineral rates, at the far end of a cell's slice,
    to 1e-9 of the network's rate constant plus the rate: ten times the free ions' bound, for reactions of up to
    eight species."""
    tp, cp = prefactors
    t = synth.random_network(N, M, 4, ionx=False, seed=synth.SEED + N)
    drawn, _, _, fine = speciated_state(t, 165, seed=M, only_ok=False)
    idx = np.flatnonzero(fine)[:131]         # the draws that speciate
    assert len(idx) > 100
    c = orc.HostCells({k: (None if v is None else v[idx].copy()) for k, v in drawn.arrays.items()}, len(idx))
    opts = dict(guess_mode=abi.PFX_GUESS_PREVIOUS, max_iterations=300)
    ref = runtime.DeviceCells.from_host(host_arrays(c), c.ncells)
    runtime.react_batch(runtime.Tables(t), ref, synth.react_opts(**opts))
    ref = ref.to_host()
    dcs = [runtime.DeviceCells.from_host(host_arrays(x), x.ncells) for x in (cp, c)]
    runtime.react_zones([runtime.Tables(tp), runtime.Tables(t)], dcs, synth.react_opts(**opts))
    out = dcs[1].to_host()
    assert np.array_equal(out["status"], ref["status"])
    solved = c.copy()
    orc.react_batch(t, solved, synth.react_opts(**opts))
    ok = (ref["status"] == 0) & (solved["status"] == 0)
    ok &= conditioning_floor(t, solved, c, synth.STEP_DT) <= 1e-11
    assert ok.sum() > 60
    rel = np.abs(out["pri_molal"][ok] - ref["pri_molal"][ok]) / ref["pri_molal"][ok]
    assert rel.max() <= 1e-10
    rate = np.abs(out["mnrl_rate"][ok] - ref["mnrl_rate"][ok])
    assert (rate <= 1e-9 * (np.abs(ref["mnrl_rate"][ok]) + t.mnrl_rate_constant)).all()
