"""The network's tiles (32 x 32, K in stages of 128) and column sums (256 rows
at a time) at the edges of their sizes, against the FP64 oracle."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,rows", [
    ((1, 1, 0, 1), 1), ((2, 1, 1, 3), 31), ((3, 33, 1, 31), 33), ((5, 127, 2, 129), 128),
    ((4, 128, 1, 256), 257), ((2, 129, 3, 17), 513), ((31, 100, 1, 1733), 65)])
def test_mlp_sizes_at_tile_edges(product, oracle, shape, rows):
    G, O = product, oracle
    rng = np.random.default_rng(rows)
    m = G.Mlp(*shape, seed=4)
    p = m.params() + 0.05 * rng.standard_normal(m.n_params).astype(np.float32)   # biases too
    m.set_params(p)
    x = rng.uniform(-1, 1, size=(rows, shape[0])).astype(np.float32)
    t = rng.normal(size=(rows, shape[3])).astype(np.float32)
    p64 = p.astype(np.float64)
    assert rel_l2(m.forward(x), O.mlp_forward(shape, p64, x.astype(np.float64))) < 1e-5
    m.set_data(x, t)
    idx = rng.permutation(rows).astype(np.int32)
    loss, g = m.loss_grad(idx)
    lw, gw = O.mlp_loss_grad(shape, p64, x[idx].astype(np.float64), t[idx].astype(np.float64))
    assert abs(loss - lw) < 1e-5 * lw
    off = 0
    for l in range(shape[2] + 1):
        ni = shape[0] if l == 0 else shape[1]
        no = shape[3] if l == shape[2] else shape[1]
        for n in (ni * no, no):
            assert rel_l2(g[off:off + n], gw[off:off + n]) < 1e-4, l
            off += n
    m.close()
