"""The fused warm start against features, network and guess in separate launches
at the ends of its 64-cell workgroups, for several networks and widths: the same
BF16 operands but for a rounding apart, so 2e-3 of the largest predicted change, as for
the default network."""
import numpy as np
import pytest

from pflotran_amd import runtime, surrogate, synth, workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,width", [(5, 1, 64), (8, 3, 128), (11, 2, 192), (15, 3, 256), (16, 4, 256)])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 193])
def test_guess(N, K, width, n):
    import torch
    t = synth.random_network(N, 2 * N, K, ionx=False, seed=synth.SEED + N)
    tab = runtime.Tables(t)
    dc, _ = workload.speciated_cells(t, tab, n)
    rng = np.random.default_rng(N + n)
    ni = 2 * N + 1 + K + 3
    mlp = surrogate.MLP((ni, width, width, N), batch_max=256, seed=3)
    for l in range(3):
        mlp.set(surrogate.W_BIAS, l, rng.normal(0, 0.3, size=mlp.dims[l + 1]))
    mlp.set_norm(rng.normal(size=ni), rng.uniform(0.05, 0.1, size=ni), rng.normal(0, 0.01, size=N), np.full(N, 20.0))
    dc.t["guess"] = torch.zeros_like(dc.t["pri_molal"])
    surrogate.guess(tab, mlp, dc)
    apart = torch.zeros_like(dc.t["guess"])
    surrogate.guess_from(mlp, mlp.forward(surrogate.features(tab, mlp, dc)), n, N, dc.t["pri_molal"], apart)
    prev = torch.log(dc.t["pri_molal"])
    a, b = torch.log(dc.t["guess"]) - prev, torch.log(apart) - prev
    assert bool(torch.isfinite(a).all())
    assert float((a - b).abs().max()) <= 2e-3 * float(b.abs().max())
