"""The reaction step's forms that its inner loop treats apart: unknowns in
ln m and in m, reactions of up to 4 and of up to 8 species, with and without ion
exchange, in each group width."""
from dataclasses import replace

import numpy as np
import pytest

import oracle as orc
from gpu_cases import conditioning_floor
from pflotran_amd import abi, runtime, synth

pytestmark = pytest.mark.gpu


def long_reactions(t):
    """The network with five to seven species in a quarter of its complexes and in a mineral: further primaries with
    coefficient 1, log K raised so that the complex stays as dilute."""
    def widen(ids, nu, logK, which):
        ids2 = np.zeros((ids.shape[0], 9), dtype=np.int32)
        nu2 = np.zeros((ids.shape[0], 8))
        ids2[:, :ids.shape[1]], nu2[:, :nu.shape[1]] = ids, nu
        logK = logK.copy()
        for i in which:
            new = [j for j in range(t.N) if j not in ids2[i, 1:1 + ids2[i, 0]]][:5 + i % 3 - ids2[i, 0]]
            for j in new:
                ids2[i, 1 + ids2[i, 0]], nu2[i, ids2[i, 0]] = j, 1.0
                ids2[i, 0] += 1
            logK[i] -= 4.0 * len(new)
        return ids2, nu2, logK
    ci, cn, ck = widen(t.cplx_specid, t.cplx_stoich, t.cplx_logK, range(0, t.M, 4))
    mi, mn, mk = widen(t.mnrl_specid, t.mnrl_stoich, t.mnrl_logK, [0])
    cZ = np.array([np.sum(cn[i, :ci[i, 0]] * t.Z[ci[i, 1:1 + ci[i, 0]]]) for i in range(t.M)])
    return replace(t, cplx_specid=ci, cplx_stoich=cn, cplx_logK=ck, cplx_Z=cZ, cplx_logKcoef=None, mnrl_specid=mi,
                   mnrl_stoich=mn, mnrl_logK=mk, mnrl_logKcoef=None, _desc=None)


@pytest.mark.parametrize("N,ionx", [(7, True), (8, False), (12, True), (15, False), (19, True)])
@pytest.mark.parametrize("use_log", [1, 0])
@pytest.mark.parametrize("long", [False, True])
def test_step_forms(N, ionx, use_log, long):
    """Status of every cell, and free ions to 1e-10 (the step's parity bound) on the cells that both bring to
    convergence and FP64 resolves to 1e-11."""
    t = synth.random_network(N, 2 * N, 2, ionx=ionx, seed=synth.SEED + 3 * N)
    if long:
        t = long_reactions(t)
    cells, _, _, _ = orc.speciated_state(t, 97)
    t = replace(t, use_log_formulation=use_log, _desc=None)
    opts = dict(guess_mode=abi.PFX_GUESS_PREVIOUS, max_iterations=300)
    ref = cells.copy()
    orc.react_batch(t, ref, synth.react_opts(**opts))
    dc = runtime.DeviceCells.from_host({k: (None if v is None else v.copy()) for k, v in cells.arrays.items()}, 97)
    runtime.react_batch(runtime.Tables(t), dc, synth.react_opts(**opts))
    out = dc.to_host()
    both = (out["status"] == 0) & (ref["status"] == 0)
    both &= conditioning_floor(t, ref, cells, synth.STEP_DT) <= 1e-11
    assert both.sum() > 25
    rel = np.abs(out["pri_molal"][both] - ref["pri_molal"][both]) / ref["pri_molal"][both]
    assert rel.max() <= 1e-10
    if use_log:
        assert np.array_equal(out["status"], ref["status"])
