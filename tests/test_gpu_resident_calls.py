"""Resident runs of few steps, as asynchronous calls make them behind a longer
one: the same state bit for bit as the same steps launched one by one."""
import numpy as np
import pytest

from test_gpu_resident import _ocean, _pair, _same

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
    for i in (0, n - 1):
        assert np.allclose(a.dissipation_series(i, 0, done), b.dissipation_series(i, 0, done), rtol=1e-12, atol=0)
    for c in (a, b):
        c.close()
