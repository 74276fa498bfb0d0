"""The warm start's training and plain inference over layer widths, batch
sizes and alignments: one launch through all layers up to 960 wide, tiled products
beyond, against the FP64 oracle with the same BF16 operand rounding: 2e-3 of the largest
entry and 1e-3 of the loss, as for the default network, and for the gradients of a few rows
2**-8 more, since one operand that FP32 and FP64 round apart is then no small
part of an entry."""
import numpy as np
import pytest

import mlp_oracle as mo
from pflotran_amd import surrogate

pytestmark = pytest.mark.gpu


def rel_to_max(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-30))


@pytest.mark.parametrize("dims,B", [
    ((40, 256, 256, 256, 15), 1), ((40, 256, 256, 256, 15), 17), ((40, 256, 256, 256, 15), 4099),
    ((33, 64, 8), 127), ((33, 50, 7), 129), ((5, 3), 16), ((1, 1), 1), ((64, 17, 130, 9, 1), 1000),
    ((40, 512, 300, 16), 515), ((257, 512, 512), 260), ((30, 513, 12), 200), ((24, 600, 520, 5), 65),
    ((9, 960, 3), 70), ((30, 961, 12), 200), ((24, 1000, 70, 5), 65)])
def test_shapes(dims, B):
    import torch
    rng = np.random.default_rng(sum(dims) + B)
    mlp = surrogate.MLP(dims, batch_max=B + 3, seed=11)
    for l in range(mlp.nlayers):
        mlp.set(surrogate.W_BIAS, l, rng.normal(0, 0.3, size=dims[l + 1]))
    # a batch that starts on a 4-byte boundary only
    xs = torch.zeros(B * dims[0] + 1, dtype=torch.float32, device="cuda")
    X = rng.normal(size=(B, dims[0])).astype(np.float32)
    T = rng.normal(size=(B, dims[-1])).astype(np.float32)
    xs[1:] = torch.from_numpy(X).cuda().ravel()
    x, y = xs[1:].view(B, dims[0]), torch.from_numpy(T).cuda()
    params = mlp.weights()
    want, _ = mo.forward(params, X, bf16=True)
    assert rel_to_max(mlp.forward(x).cpu().numpy(), want) <= 2e-3
    tol = 2e-3 + (2.0 ** -8 if B < 64 else 0.0)
    loss, grads = mo.loss_and_grads(params, X, T, bf16=True)
    for step in range(2):                       # gradients alone, then with the update
        got = mlp.train_step(x, y, 1e-3, want_loss=True) if step else mlp.gradients(x, y)
        assert abs(got - loss) <= 1e-3 * loss
        for g, w in zip(mlp.gradients_host(), grads):
            assert rel_to_max(g[0], w[0]) <= tol and rel_to_max(g[1], w[1]) <= tol
    # the next pass reads the updated weights
    new = mlp.weights()
    for (w0, b0), (w1, b1), (gw, gb) in zip(params, new, mlp.gradients_host()):
        for p0, p1, g in ((w0, w1, gw), (b0, b1, gb)):
            q, _, _ = mo.adam_step(p0.astype(np.float64), g.astype(np.float64), 0.0, 0.0, 1, 1e-3)
            assert np.max(np.abs(p1 - q)) <= 1e-6
    want, _ = mo.forward(new, X, bf16=True)
    assert rel_to_max(mlp.forward(x).cpu().numpy(), want) <= 2e-3
