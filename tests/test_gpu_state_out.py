"""State and output calls through the pinned staging buffer (2 MB, in
quarters when the output is larger): whole, in reference order, at sizes
below, at the edge of and above the buffer."""
import numpy as np
import pytest

from conftest import generated_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,precision", [(3, 0), (5, 1), (6, 0), (7, 0), (7, 1), (8, 0)])
def test_outputs_are_the_state_in_reference_order(product, level, precision):
    G = product
    g, _ = generated_grid(level)
    mesh = G.Mesh(g, 252.1e3)
    p, _ = G.make_params(time_step=1.0)
    held = np.float32 if precision else np.float64
    rng = np.random.default_rng(level)
    v = rng.standard_normal(mesh.E).astype(held).astype(float)
    eta = rng.standard_normal(mesh.N).astype(held).astype(float)
    dv = rng.standard_normal((mesh.E, 3)).astype(held).astype(float)
    de = rng.standard_normal((mesh.N, 3)).astype(held).astype(float)
    c = G.Context(mesh, [p, p], precision=precision)
    c.set_state(1, v=v, dvdt=dv, eta=eta, detadt=de, iter=5)
    s = c.get_state(1)
    assert np.array_equal(s["v"], v) and np.array_equal(s["eta"], eta)
    # after step 4 the rows are (f, f, the one before): entries 1 and 2 as set
    assert np.array_equal(s["dvdt"], dv[:, [1, 1, 2]]) and np.array_equal(s["detadt"], de[:, [1, 1, 2]])
    rp, col, val = mesh.rbf_operator()
    want = np.add.reduceat(val * v[col], rp[:-1])
    c.set_rbf()
    assert np.allclose(c.velocity_xyz(1).ravel(), want, rtol=0, atol=1e-12 * np.abs(val).max())
    # the tangential part: orthogonal to the normal one, the same TRiSK sum as on the host
    n = mesh.get("face_normal").reshape(-1, 2)
    uv = c.velocity_en(1)
    assert np.allclose((uv * n).sum(1), v * (n * n).sum(1), rtol=0, atol=1e-6 if precision else 1e-12)
    cnt, fr, w = mesh.get("interp_count"), mesh.get("interp_friends").reshape(-1, 10), mesh.get("interp_weights")
    coef = w.reshape(-1, 10) * mesh.get("face_len")[np.maximum(fr, 0)] / mesh.get("face_node_dist")[:, None]
    vt = np.where(np.arange(10) < cnt[:, None], coef * v[np.maximum(fr, 0)], 0.0).sum(1)
    got = uv[:, 0] * n[:, 1] - uv[:, 1] * n[:, 0]
    assert np.allclose(got, vt * (n * n).sum(1), rtol=0, atol=1e-5 if precision else 1e-12)
    c.close()
