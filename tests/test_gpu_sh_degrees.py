"""The on-the-fly projection at degrees with and without a compiled kernel:
coefficients and synthesis against the dense least-squares fit in FP64."""
import numpy as np
import pytest

from conftest import generated_grid, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("level,degree", [(4, 0), (4, 1), (4, 5), (5, 8), (5, 9), (5, 12), (6, 16), (5, 17), (6, 20),
                                          (6, 24), (5, 25), (6, 31), (6, 32), (6, 33)])
def test_projection_and_synthesis(product, level, degree):
    G = product
    g, arrs = generated_grid(level)
    mesh = G.Mesh(g, 252.1e3)
    p, _ = G.make_params(time_step=1.0)
    Y = G.sh_basis(degree, arrs["lat"], arrs["lon"])
    field = np.random.default_rng(degree).standard_normal(mesh.N)
    want = np.linalg.solve(Y.T @ Y, Y.T @ field)
    c = G.Context(mesh, p)
    c.set_sh(degree, np.ones(degree + 1), mode=G.SH_RECUR)
    got = c.sh_project(field)
    # sums of N terms and a recurrence of `degree` steps in 53 bits
    assert rel_l2(got, want) < 1e-12
    assert rel_l2(c.sh_synthesize(want), Y @ want) < 1e-12
    c.close()


@pytest.mark.parametrize("precision,level,degree,n", [(0, 6, 12, 1), (1, 6, 12, 1), (1, 5, 20, 3), (0, 5, 7, 2)])
def test_coupled_step_in_the_next_degrees_kernel(product, oracle, precision, level, degree, n):
    """A step coupled to a degree that runs in a larger degree's kernel
    against the stored FP64 basis."""
    G = product
    g, _ = generated_grid(level)
    mesh = G.Mesh(g, 232.1e3)
    beta = G.surface_beta(G.LID_MEMBR, degree, 252.1e3, 0.113, 5e3, 38e3)
    p, _ = G.make_params(radius=232.1e3, g=0.1166, surface=G.LID_MEMBR, shell_thickness=5e3, time_step=2.0)
    out = []
    for prec, mode in ((precision, G.SH_RECUR), (0, G.SH_FP64)):
        c = G.Context(mesh, [p] * n, precision=prec)
        c.set_sh(degree, beta, mode=mode)
        c.step(40)
        out.append(c.get_state(n - 1))
        c.close()
    tol = 1e-10 if precision == 0 else 1e-4
    for k in ("v", "eta", "dvdt"):
        assert rel_l2(out[0][k], out[1][k]) < tol, k


@pytest.mark.parametrize("level,n_many,degree", [(4, 130, 9), (4, 130, 15), (4, 130, 16), (5, 40, 24), (5, 40, 31),
                                                 (5, 40, 32)])
def test_coupled_step_of_many_and_one(product, level, n_many, degree):
    """A batch large enough for four synthesis waves per workgroup against
    one instance, which runs eight: the same sums in another order, 20 steps."""
    G = product
    g, _ = generated_grid(level)
    mesh = G.Mesh(g, 232.1e3)
    beta = G.surface_beta(G.LID_MEMBR, degree, 252.1e3, 0.113, 5e3, 38e3)
    p, _ = G.make_params(radius=232.1e3, g=0.1166, surface=G.LID_MEMBR, shell_thickness=5e3, time_step=2.0)
    out = []
    for n in (1, n_many):  # 6 and 780, 21 and 840 workgroups
        c = G.Context(mesh, [p] * n)
        c.set_sh(degree, beta, mode=G.SH_RECUR)
        c.step(20)
        out.append(c.get_state(n - 1))
        c.close()
    for k in ("v", "eta", "dvdt"):
        assert rel_l2(out[1][k], out[0][k]) < 1e-10, k
