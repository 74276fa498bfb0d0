"""Workgroups of a zoned launch: a default split never has more than one zone
alone (all that are resident), and a plan of more workgroups than that does
every cell once, with the bits of the default split."""
import numpy as np
import pytest

from gpu_cases import host_arrays, speciated_state
from pflotran_amd import abi, runtime, synth

pytestmark = pytest.mark.gpu
FIELDS = ("pri_molal", "total", "sec_molal", "mnrl_rate", "num_iterations", "status")


@pytest.fixture(scope="module")
def zone():
    t = synth.random_network(15, 30, 2, ionx=False, seed=synth.SEED + 2)
    cells, _, _, _ = speciated_state(t, 61)

    def batch(n):
        idx = np.arange(n) % 61
        return runtime.DeviceCells.from_host({k: (None if v is None else v[idx].copy())
                                              for k, v in host_arrays(cells).items()}, n)
    return t, batch


@pytest.mark.parametrize("variant", [0, 1, 2])
def test_default_split_is_resident(zone, variant):
    t, batch = zone
    opts = synth.react_opts(guess_mode=abi.PFX_GUESS_PREVIOUS)

    def total(nzones):
        plan = abi.ZonePlan()
        plan.nzones, plan.variant = nzones, variant
        tabs = [runtime.Tables(t) for _ in range(nzones)]
        _, _, plan = runtime.react_zones(tabs, [batch(40003) for _ in range(nzones)], opts, plan)
        return sum(plan.blocks[z] for z in range(nzones))
    alone = total(1)
    for nzones in (2, 3, 5, 6, 7, 8):
        assert alone - nzones < total(nzones) <= alone


@pytest.mark.parametrize("factor", [1, 2, 5])
def test_plans_beyond_residency(zone, factor):
    import torch
    t, batch = zone
    opts = synth.react_opts(guess_mode=abi.PFX_GUESS_PREVIOUS)
    sizes = (30011, 9001, 17)
    tabs = [runtime.Tables(t) for _ in sizes]
    dcs = [batch(n) for n in sizes]
    _, st, plan = runtime.react_zones(tabs, dcs, opts)
    for z in range(3):
        plan.blocks[z] *= factor
    again = [batch(n) for n in sizes]
    _, st2, used = runtime.react_zones(tabs, again, opts, plan)
    for z, n in enumerate(sizes):
        for k in FIELDS:
            assert torch.equal(again[z].t[k], dcs[z].t[k]), (z, k)
        assert st2[z].total_iterations == st[z].total_iterations == int(dcs[z].t["num_iterations"].sum())
        assert used.blocks[z] <= max(1, (n + 15) // 16)
