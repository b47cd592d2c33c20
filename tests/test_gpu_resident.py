"""The resident step (many steps per launch, the ocean held on the chip)
against the same steps launched one by one: the same state bit for bit."""
import threading

import numpy as np
import pytest

from conftest import generated_grid

pytestmark = pytest.mark.gpu

KEYS = ("v", "eta", "dvdt", "detadt")


def _ocean(G, level, n, tide="FULL", quad=False, **kw):
    g, _ = generated_grid(level)
    rng = np.random.default_rng(level * 100 + n)
    ts = 0.3 / (0.0193 * (g.n / 10242.0) ** 0.5)
    extra = dict(semimajor=671100000.0) if tide == "PLANET" else {}
    if quad:
        extra.update(friction=G.QUADRATIC, quad_drag=1, alpha=2e-3)
    ps = [G.make_params(time_step=ts, h=float(10 ** rng.uniform(3.5, 4.6)), tide=getattr(G, tide),
                        obliquity=float(np.radians(rng.uniform(0, 1))), **{**extra, **kw})[0] for _ in range(n)]
    mesh = G.Mesh(g, ps[0].radius)
    start = [(1e-3 * rng.standard_normal(mesh.E), 1e-2 * rng.standard_normal(mesh.N)) for _ in range(n)]
    return mesh, ps, start


def _pair(G, mesh, ps, start, precision, patches=1):
    out = []
    for opt in (patches, 0):
        c = G.Context(mesh, ps, precision=precision)
        c.set_option(G.OPT_RESIDENT, opt)
        for b, (v, eta) in enumerate(start):
            c.set_state(b, v=v, eta=eta)
        out.append(c)
    return out


def _same(a, b, insts):
    for i in insts:
        x, y = a.get_state(i), b.get_state(i)
        assert x["iter"] == y["iter"]
        for k in KEYS:
            assert np.array_equal(x[k], y[k]), (i, k)


# (level, precision, instances, patches per instance (1: automatic), tide, quadratic drag): the kernel
# variants and their edges -- one patch (no messages), patches of 40 cells, more instances than fit at
# once (rounds, an uneven last one), no tide, 7 tide fields, two workgroups per CU
@pytest.mark.parametrize("level,precision,n,patches,tide,quad", [
    (3, 0, 1, 1, "ECC", False), (4, 0, 1, 2, "ECC", False), (4, 0, 1, 40, "FULL2", False),
    (4, 1, 1, 16, "NONE", False), (5, 0, 1, 5, "PLANET", True), (5, 1, 3, 7, "FULL2", True),
    (6, 0, 1, 1, "FULL", False), (6, 0, 23, 1, "OBLIQ", False), (6, 1, 33, 32, "FULL", True),
    (4, 0, 201, 2, "FULL", False), (5, 1, 131, 4, "FULL", False), (7, 1, 5, 1, "ECC", False),
    (7, 0, 1, 1, "FULL", True), (8, 0, 1, 1, "FULL2", True), (8, 1, 2, 1, "FULL", False)])
def test_resident_steps_equal_single_launches(product, level, precision, n, patches, tide, quad):
    G = product
    mesh, ps, start = _ocean(G, level, n, tide, quad)
    a, b = _pair(G, mesh, ps, start, precision, patches)
    insts = sorted({0, n // 2, n - 1})
    done = 0
    for steps in (4, 9, 1, 30):     # both Euler steps, an odd run, a single launch between two runs
        for c in (a, b):
            c.step(steps, sync=False)
        done += steps
        _same(a, b, insts)
    for i in insts:
        x, y = a.dissipation_series(i, 0, done), b.dissipation_series(i, 0, done)
        assert np.allclose(x, y, rtol=1e-12, atol=0)
    assert np.allclose(a.dissipation(), b.dissipation(), rtol=1e-12, atol=0)
    for c in (a, b):
        c.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_resident_long_run_state_changes_and_sampled_steps(product, precision):
    """Across launches (more steps than one launch takes), a set_state of one
    instance in mid-run, AB3 from step 0, a retirement, and runs cut by
    steps sampled for timing."""
    G = product
    mesh, ps, start = _ocean(G, 4, 4, init_load=1)
    a, b = _pair(G, mesh, ps, start, precision)
    for c in (a, b):
        c.step(2311)
    _same(a, b, range(4))
    st = b.get_state(2)
    for c in (a, b):
        c.set_state(1, st["v"], st["dvdt"], st["eta"], st["detadt"], 7)
        c.step(50)
        c.retire([0, 1, 3])
        c.step(50)
        c.enable_timing(16)
        c.step(75)
    _same(a, b, range(3))
    assert a.timing()["step_ms"] > 0
    x, y = (c.orbit_stats([0, 2], [100, 60]) for c in (a, b))
    assert np.allclose(x[:, 0], y[:, 0], rtol=1e-12, atol=0)
    for c in (a, b):
        c.close()


def test_resident_launches_of_two_contexts(product):
    """Two contexts stepping from two threads, their launches in flight at
    the same time: each ends as it does alone."""
    G = product
    mesh, ps, start = _ocean(G, 6, 2)
    one = [G.Context(mesh, [p]) for p in ps]
    want = []
    for c, (v, eta) in zip(one, start):
        c.set_state(v=v, eta=eta)
        for _ in range(6):
            c.step(40)
        want.append(c.get_state())
        c.set_state(v=v, eta=eta, dvdt=np.zeros((mesh.E, 3)), detadt=np.zeros((mesh.N, 3)))

    def go(c):
        for _ in range(6):
            c.step(40, sync=False)
        c.sync()
    th = [threading.Thread(target=go, args=(c,)) for c in one]
    for t in th:
        t.start()
    for t in th:
        t.join(60)
        assert not t.is_alive()
    for c, w in zip(one, want):
        got = c.get_state()
        for k in KEYS:
            assert np.array_equal(got[k], w[k]), k
        c.close()
