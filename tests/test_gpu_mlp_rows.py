"""Plain inference of narrow networks around the batch sizes where the kernel
gets fewer wavefronts, and one narrow layer around those where it is a plain
product: against the FP64 oracle with the same BF16 operand rounding (2e-3 of the
largest entry, as for the default network), and a large batch bit for bit as its
pieces."""
import numpy as np
import pytest

import mlp_oracle as mo
from pflotran_amd import surrogate
from test_gpu_call_costs import least

pytestmark = pytest.mark.gpu
RESIDENT = 16384


def network(dims, bmax, seed=3):
    rng = np.random.default_rng(seed)
    m = surrogate.MLP(dims, batch_max=bmax, seed=seed)
    for l in range(m.nlayers):
        m.set(surrogate.W_BIAS, l, rng.normal(0, 0.3, size=dims[l + 1]))
    return m


@pytest.mark.parametrize("dims", [(4, 16, 1), (32, 32, 32), (33, 20, 7), (16, 64, 64, 16), (40, 65, 15), (5, 128, 3),
                                  (129, 8, 2), (40, 256, 9), (4, 1), (63, 32), (64, 33), (128, 16)])
@pytest.mark.parametrize("extra", [0, 1, 30])
def test_batches_around_the_resident_rows(dims, extra):
    import torch
    one = len(dims) == 2 and dims[1] <= 32
    n = RESIDENT * (max(1, dims[0] // 64) if one else 1) + extra
    m = network(dims, n)
    x = torch.randn((n, dims[0]), device="cuda", generator=torch.Generator("cuda").manual_seed(sum(dims)))
    y = m.forward(x)
    want, _ = mo.forward(m.weights(), x.cpu().numpy(), bf16=True)
    assert np.max(np.abs(y.cpu().numpy() - want)) <= 2e-3 * np.max(np.abs(want))
    if not one:
        assert torch.equal(y, torch.cat([m.forward(x[k:k + 9000]) for k in range(0, n, 9000)]))


def test_narrow_networks_cost_less_than_wide_ones():
    """262144 rows: a sixteenth of the products took 0.55, one layer 0.18 of the time."""
    import torch
    n = 262144
    x40, x4 = torch.randn((n, 40), device="cuda"), torch.randn((n, 4), device="cuda")
    wide, narrow, one = network((40, 256, 256, 15), n), network((40, 64, 64, 15), n), network((4, 1), n)
    t = least(lambda: wide.forward(x40))
    assert least(lambda: narrow.forward(x40)) <= 0.42 * t
    assert least(lambda: one.forward(x4)) <= 0.12 * t
