"""Resident runs of few steps, as asynchronous calls make them behind a longer
one: the same state bit for bit as the same steps launched one by one."""
import threading

import numpy as np
import pytest

from test_gpu_resident import KEYS, _ocean, _pair, _same

pytestmark = pytest.mark.gpu


# (level, precision, instances, patches per instance (1: automatic), AB3 from step 0): one instance and
# several rounds of instances, where runs of 1, 2 and 3 steps send no, one and two messages per slot
@pytest.mark.parametrize("level,precision,n,patches,load", [
    (4, 0, 1, 1, 0), (6, 1, 1, 1, 1), (4, 0, 201, 2, 0), (5, 1, 131, 4, 1), (7, 0, 3, 1, 0)])
def test_runs_of_few_steps(product, level, precision, n, patches, load):
    G = product
    mesh, ps, start = _ocean(G, level, n, "FULL", init_load=load)
    a, b = _pair(G, mesh, ps, start, precision, patches)
    done = 0
    for calls in ((6, 1, 2, 3, 7, 1), (4, 2, 1, 1, 9, 3)):
        for steps in calls:
            a.step(steps, sync=False)
        b.step(sum(calls))
        done += sum(calls)
        _same(a, b, sorted({0, n // 2, n - 1}))
    assert a.option(G.OPT_RESIDENT_ACTIVE) > 0
    for i in (0, n - 1):
        assert np.allclose(a.dissipation_series(i, 0, done), b.dissipation_series(i, 0, done), rtol=1e-12, atol=0)
    for c in (a, b):
        c.close()


# (level, precision, instances, option, tide, quadratic drag) -> patches (None: any).  One patch, which has
# no messages: 162 cells when the chip holds one workgroup per instance; one workgroup of 512 and of 1024
# lanes; patches at the limit of 641 cells and of the LDS (4 tide fields in FP64, 7 in FP32)
@pytest.mark.parametrize("level,precision,n,option,tide,quad,patches", [
    (3, 0, 129, 1, "FULL", False, 1), (3, 1, 300, 1, "FULL2", True, None), (2, 0, 3, 1, "ECC", False, 1),
    (4, 0, 1, 1, "ECC", False, 16), (4, 0, 1, 2, "FULL2", True, 2), (5, 1, 1, 5, "PLANET", False, 5),
    (6, 0, 23, 1, "OBLIQ", False, None), (8, 0, 1, 1, "FULL", True, 256), (8, 1, 1, 1, "FULL2", True, 256)])
def test_the_resident_step_runs(product, level, precision, n, option, tide, quad, patches):
    G = product
    mesh, ps, start = _ocean(G, level, n, tide, quad)
    a, b = _pair(G, mesh, ps, start, precision, option)
    for steps in (7, 30):
        for c in (a, b):
            c.step(steps)
        in_use = a.option(G.OPT_RESIDENT_ACTIVE)
        assert (in_use == patches if patches else in_use > 0) and b.option(G.OPT_RESIDENT_ACTIVE) == 0
        _same(a, b, sorted({0, n // 2, n - 1}))
    for c in (a, b):
        c.close()


# the launch that waits in vain for a workgroup, with and without steps sampled for timing: single oceans,
# rounds of instances, a batch whose single steps are interleaved
@pytest.mark.parametrize("level,precision,n,miss,stride", [
    (4, 0, 1, 1, 0), (4, 0, 1, 2, 0), (6, 1, 1, 2, 16), (4, 0, 201, 1, 0), (7, 1, 16, 2, 0), (8, 0, 1, 1, 16)])
def test_a_launch_taken_back(product, level, precision, n, miss, stride):
    """Steps of a launch taken back, and of those queued behind it, are
    stepped again singly; the resident step runs again when asked for."""
    G = product
    mesh, ps, start = _ocean(G, level, n, "FULL")
    a, b = _pair(G, mesh, ps, start, precision)
    for c in (a, b):
        c.enable_timing(stride)
    a.set_option(G.OPT_RESIDENT_MISS, miss)
    done = 0
    for again in (False, True):
        for steps in (30, 41, 3, 17):
            a.step(steps, sync=False)
            b.step(steps)
            done += steps
        _same(a, b, sorted({0, n // 2, n - 1}))
        assert (a.option(G.OPT_RESIDENT_ACTIVE) > 0) == again
        a.set_option(G.OPT_RESIDENT, 1)
    for i in (0, n - 1):
        assert np.allclose(a.dissipation_series(i, 0, done), b.dissipation_series(i, 0, done), rtol=1e-12, atol=0)
    for c in (a, b):
        c.close()


def test_launches_side_by_side(product):
    """Contexts of several sizes stepping from threads of their own, their
    launches beside and behind each other: each ends as it does alone, and none
    of them is taken back."""
    G = product
    runs = []
    for level, option, steps in [(4, 1, 37), (4, 1, 40), (5, 1, 25), (6, 200, 30), (6, 1, 20), (5, 50, 33), (4, 3, 50),
                                 (7, 1, 15)]:
        mesh, ps, start = _ocean(G, level, 1)
        c = G.Context(mesh, ps)
        c.set_option(G.OPT_RESIDENT, option)
        c.set_state(v=start[0][0], eta=start[0][1])
        runs.append((c, mesh, start[0], steps))
    want = []
    for c, mesh, (v, eta), steps in runs:
        for _ in range(12):
            c.step(steps)
        want.append(c.get_state())
        c.set_state(v=v, eta=eta, dvdt=np.zeros((mesh.E, 3)), detadt=np.zeros((mesh.N, 3)))

    def go(c, steps):
        for k in range(12):
            c.step(steps, sync=False)
            if k % 5 == 4:
                c.sync()
        c.sync()
    th = [threading.Thread(target=go, args=(c, steps)) for c, _, _, steps in runs]
    for t in th:
        t.start()
    for t in th:
        t.join(60)
        assert not t.is_alive()
    for (c, _, _, _), w in zip(runs, want):
        assert c.option(G.OPT_RESIDENT_ACTIVE) > 0
        got = c.get_state()
        for k in KEYS:
            assert np.array_equal(got[k], w[k]), k
        c.close()
