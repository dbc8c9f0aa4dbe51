"""GPU gradients against the FP64 oracle at the edges of the training kernels'
row tiles: less than a tile, one row past a tile and past a 32-row block, the
last batch of the 16-row tiles and the first of the 32-row ones, in this order
on one network, whose buffers a larger batch sizes for a smaller one after it."""
import numpy as np
import pytest

from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1, 15, 17, 33), (8193, 8192, 8161)])
def test_gradients_at_tile_edges(gpu, sizes):
    from anacor_public_amd import _lib
    from anacor_public_amd.surrogate import MLP
    rng = np.random.default_rng(5)
    P = np.concatenate([rng.uniform(-1, 1, b - a).astype(np.float32) / np.sqrt(f) for a, b, f in
                        [(a, b, _lib.MLP_INPUTS if name in ("W1", "b1") else 256)
                         for name, (a, b, _) in MO.offsets().items()]])
    with MLP(seed=1) as m:
        m.set_params(P)
        for n in sizes:
            X = rng.uniform(-1, 1, size=(n, _lib.MLP_INPUTS)).astype(np.float32)
            t = rng.normal(size=n).astype(np.float32)
            g, loss = m.gradients(X, t)
            yo, cache = MO.forward(P, X.astype(np.float64), bf16=True)
            go, losso = MO.backward(cache, yo, t.astype(np.float64))
            assert loss == pytest.approx(losso, rel=1e-5)
            for name, (a, b, _) in MO.offsets().items():
                rel = np.linalg.norm(g[a:b] - go[a:b]) / np.linalg.norm(go[a:b])
                assert rel < 1e-4, (n, name, rel)
