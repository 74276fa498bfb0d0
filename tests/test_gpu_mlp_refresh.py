"""The warm start's products read the weights that are set, whatever came
between: a captured pass that has not been replayed, weights set between
replays, passes on another stream than the first.  Each is compared bit for bit
with a network made with those weights."""
import numpy as np
import pytest

from pflotran_amd import surrogate, synth, workload, runtime

pytestmark = pytest.mark.gpu
DIMS = (40, 64, 128, 15)


def drawn(seed):
    rng = np.random.default_rng(seed)
    return [rng.normal(0, 0.2, size=(n, k)).astype(np.float32) for k, n in zip(DIMS, DIMS[1:])]


def network(weights):
    mlp = surrogate.MLP(DIMS, batch_max=512, seed=1)
    for l, w in enumerate(weights):
        mlp.set(surrogate.W_WEIGHT, l, w)
    return mlp


def rows(seed, n=200):
    import torch
    rng = np.random.default_rng(seed)
    dev = lambda *s: torch.from_numpy(rng.normal(size=s).astype(np.float32)).cuda()  # noqa: E731
    return dev(n, DIMS[0]), dev(n, DIMS[-1])


def raw_gradients(mlp, x, y):
    """Gradients without reading the loss back, as a captured step asks for them."""
    import torch
    rc = runtime.load_library().pfx_mlp_gradients(mlp.handle, x.data_ptr(), y.data_ptr(), x.shape[0], None,
                                                  torch.cuda.current_stream().cuda_stream)
    assert rc == 0


def same(a, b):
    return all(np.array_equal(p, q) for u, v in zip(a, b) for p, q in zip(u, v))


def test_eager_pass_after_a_capture():
    """A capture enqueues nothing: the eager pass after it stands on its own."""
    import torch
    x, y = rows(3)
    mlp = network(drawn(5))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        mlp.forward(x)
    got = mlp.forward(x)
    assert torch.equal(got, network(drawn(5)).forward(x))


def test_replays_follow_the_weights():
    import torch
    x, y = rows(4)
    mlp = network(drawn(6))
    out = mlp.forward(x)                    # the state that a program captures in
    graph, gradients = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = mlp.forward(x)
    with torch.cuda.graph(gradients):
        raw_gradients(mlp, x, y)
    for seed in (7, 8, 9):
        new = drawn(seed)
        for l, w in enumerate(new):
            mlp.set(surrogate.W_WEIGHT, l, w)
        ref = network(new)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref.forward(x))
        gradients.replay()
        torch.cuda.synchronize()
        raw_gradients(ref, x, y)
        assert same(mlp.gradients_host(), ref.gradients_host())


def test_captured_guess_follows_the_weights():
    """The fused warm start, captured before its first eager use."""
    import torch
    t = synth.random_network(15, 50, 3, ionx=True)
    tab = runtime.Tables(t)
    dc, _ = workload.speciated_cells(t, tab, 130)
    dc.t["guess"] = torch.zeros_like(dc.t["pri_molal"])
    mlp = network(drawn(10))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        surrogate.guess(tab, mlp, dc)
    for seed in (10, 11, 12):
        new = drawn(seed)
        for l, w in enumerate(new):
            mlp.set(surrogate.W_WEIGHT, l, w)
        surrogate.guess(tab, network(new), dc)
        want = dc.t["guess"].clone()
        dc.t["guess"].zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(dc.t["guess"], want)
        dc.t["guess"].zero_()
        surrogate.guess(tab, mlp, dc)
        torch.cuda.synchronize()
        assert torch.equal(dc.t["guess"], want)


def test_passes_on_two_streams():
    """Weights set, then a pass on one stream held up behind other work and one on a second stream."""
    import torch
    x, _ = rows(5)
    want = network(drawn(13)).forward(x)
    mlp = network(drawn(14))
    mlp.forward(x)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    big = torch.randn(6000, 6000, device="cuda")
    for l, w in enumerate(drawn(13)):
        mlp.set(surrogate.W_WEIGHT, l, w)
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        for _ in range(8):
            big = big @ big * 1e-4
        first = mlp.forward(x)
    with torch.cuda.stream(b):
        second = mlp.forward(x)
    torch.cuda.synchronize()
    assert torch.equal(first, want) and torch.equal(second, want)


def test_streams_after_training():
    """Weights that a training step has moved, read on another stream after it."""
    import torch
    x, y = rows(6)
    mlp = network(drawn(15))
    mlp.train_step(x, y, 1e-2)
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        got = mlp.forward(x)
    torch.cuda.synchronize()
    ref = surrogate.MLP(DIMS, batch_max=512, seed=1)
    for l, (w, b) in enumerate(mlp.weights()):
        ref.set(surrogate.W_WEIGHT, l, w)
        ref.set(surrogate.W_BIAS, l, b)
    assert torch.equal(got, ref.forward(x))
