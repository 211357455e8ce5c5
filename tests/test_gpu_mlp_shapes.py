"""The network's matrix-core products at the sizes where a tile or a range of
rows can go wrong: ragged and single rows, widths that are no multiple of 4
(scalar loads) or of the tile, and row counts at the edges of the weight
gradients' ranges, against the float64 statement of the same network
(oracle/mlp.py).

Tolerance: each result is a chain of at most five FP32 products of inner
length k <= 200 (the row sums: blocks of at most 128 rows), whose relative
error is below k eps = 200 x 6e-8 = 1.2e-5 per product against the norm of
the terms, so 1e-4 of the block's norm bounds it (and 1e-5 of the largest
output covers the forward pass)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,width,n_out", [(200, 128, 16), (13, 37, 5), (64, 100, 33), (7, 130, 1)])
@pytest.mark.parametrize("rows", [1, 63, 65, 128, 129, 1000, 4161, 8200])
def test_gradient_at_tile_and_range_edges(ctx, n_in, width, n_out, rows):
    from oracle import mlp
    rng = np.random.default_rng(rows * 1000 + n_in)
    ctx.mlp_create(n_in, width, n_out, 5)
    dims = [(n_in, width), (width, width), (width, width), (width, n_out)]
    p = np.concatenate([np.concatenate([rng.uniform(-1, 1, a * b) * np.sqrt(6.0 / (a + b)), rng.normal(0, 0.1, b)])
                        for a, b in dims]).astype(np.float32)
    ctx.mlp_params(set_to=p)
    X = rng.standard_normal((rows, n_in)).astype(np.float32)
    T = rng.standard_normal((rows, n_out)).astype(np.float32)
    Mk = (rng.uniform(size=(rows, n_out)) < 0.7).astype(np.float32)
    loss, g = ctx.mlp_gradient(X, T, Mk)
    L, gr = mlp.loss_grad(p, X, T, Mk, n_in, width, n_out)
    assert abs(loss - L) <= 1e-5 * L
    o = 0
    for a, b in dims:
        for size in (a * b, b):
            sl = slice(o, o + size)
            assert np.linalg.norm(g[sl] - gr[sl]) <= 1e-4 * np.linalg.norm(gr[sl]) + 1e-9
            o += size
    Y = ctx.mlp_forward(X, n_out)
    Yr = mlp.forward(p, X, n_in, width, n_out)
    assert np.max(np.abs(Y - Yr)) <= 1e-5 * max(1.0, np.max(np.abs(Yr)))
