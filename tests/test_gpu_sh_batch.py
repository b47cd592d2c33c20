"""FP64 shells by recurrence: an instance's trajectory does not depend on the
rest of its batch, bit for bit."""
import numpy as np
import pytest

from conftest import generated_grid

pytestmark = pytest.mark.gpu


# (level, degree, instances, cells per lane of the analysis; 0: automatic).  Batches on both sides of
# the synthesis' limit of eight waves per workgroup and, at degrees without a kernel of their own, of
# the analysis' automatic cells per lane
@pytest.mark.parametrize("level,degree,n,cells", [
    (4, 9, 130, 0), (5, 12, 40, 0), (6, 12, 40, 0), (6, 20, 24, 0), (6, 31, 12, 0), (5, 16, 40, 4), (6, 32, 12, 8),
    (5, 8, 40, 4), (5, 33, 12, 0)])
def test_fp64_shells_alone_and_in_batch(product, level, degree, n, cells):
    G = product
    g, _ = generated_grid(level)
    mesh = G.Mesh(g, 232.1e3)
    rng = np.random.default_rng(degree)
    ps, betas = [], []
    for _ in range(n):
        h = float(10 ** rng.uniform(3.5, 4.6))
        ps.append(G.make_params(radius=232.1e3, g=0.1166, surface=G.LID_MEMBR, shell_thickness=20e3, love_reduct=0.99,
                                h=h, time_step=2.0)[0])
        betas.append(G.surface_beta(G.LID_MEMBR, degree, 252.1e3, 0.113, 20e3, h))
    start = [(1e-3 * rng.standard_normal(mesh.E), 1e-2 * rng.standard_normal(mesh.N)) for _ in range(n)]

    def run(which):
        c = G.Context(mesh, [ps[b] for b in which])
        c.set_option(G.OPT_SH_CELLS, cells)
        c.set_sh(degree, np.stack([betas[b] for b in which]), mode=G.SH_RECUR)
        for k, b in enumerate(which):
            c.set_state(k, v=start[b][0], eta=start[b][1])
        c.step(6)
        out = [c.get_state(k) for k in range(len(which))]
        c.close()
        return out
    batch = run(range(n))
    for b in (0, n // 2, n - 1):
        (one,) = run([b])
        for k in ("v", "eta", "dvdt", "detadt"):
            assert np.array_equal(one[k], batch[b][k]), (b, k)
