"""The launch forms a call's sizes choose between, at the sizes where a form
begins, ends or has a remainder, against the CPU oracle or plain numpy."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(77)


@pytest.mark.parametrize("n_ops", [1, 2, 4, 5, 9])
def test_short_graph_replays(ggml, gpu, n_ops):
    """a graph of a few launches, replayed (launch by launch up to four, as
    one HIP graph beyond): every compute is on the inputs of that compute.
    Scaling by a power of two is exact."""
    print(f"short graph of {n_ops}", flush=True)
    G = ggml.Graph()
    X = G.new(ggml.F32, 1000, 3)
    y, f = X, 1.0
    for i in range(n_ops):
        s = 2.0 if i % 2 else -0.25
        y, f = G.lib.ggml_scale(G.ctx, y, s), f * s
    G.build(y)
    G.allocate(gpu.buft)
    for it in range(6):
        x = RNG.standard_normal((3, 1000)).astype(np.float32)
        G.set(X, x)
        assert G.compute(gpu.backend) == 0
        assert np.array_equal(G.get(y).reshape(3, 1000), x * np.float32(f))
    G.free()
