"""Host logic of the resident step without a GPU: the library runs on a stub
of the HIP runtime (hip_stub.cpp) in a process of its own.  The stub's kernels
compute nothing; what is checked is which launches are made, what an entry
point returns, and what it holds."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

from conftest import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))
PRELUDE = """
import ctypes, functools, sys
S = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
S.stub_log.restype = ctypes.c_char_p
S.stub_device_bytes.restype = ctypes.c_size_t
S.stub_fail_allocations_of.argtypes = [ctypes.c_size_t]
S.stub_end_resident.argtypes = [ctypes.c_int, ctypes.c_uint]
import numpy as np
import geodesicodis_amd as G

def log():
    out = S.stub_log().decode().split("\\n")[:-1]
    S.stub_clear()
    return out

def steps(lines, kind="step"):
    return [int(x.split()[1]) for x in lines if x.startswith(kind + " ")]

def runs(lines):
    return sum(x.startswith("resident ") for x in lines)

@functools.lru_cache(None)
def mesh(level=4):
    return G.Mesh(G.Grid.generate(level, 64), 252.1e3)

def ocean(n=1, level=4, precision=0, **kw):
    p = G.make_params(time_step=1.0, **kw)[0]
    return G.Context(mesh(level), [p] * n, precision=precision)

def refused(call):
    try:
        call()
    except G.OdisError as e:
        return e.code
    return 0
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    so = tmp_path_factory.mktemp("stub") / "hip_stub.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_stub.cpp"), "-o", str(so)], check=True)

    def run(body):
        r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), str(so)], cwd=ROOT, timeout=120,
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


@pytest.mark.parametrize("stride", [0, 16])
def test_steps_of_a_launch_taken_back_are_stepped_once_each(stub, stride):
    """The first launch, or the second of a timed run, is taken back: every
    step from there on is launched singly, once, and the call goes on so."""
    stub("""
    c = ocean()
    if %d:
        c.enable_timing(%d)
    c.step(1)          # a first single step, then runs
    log()
    S.stub_end_resident(%d, 0)
    c.step(100)
    lines = log()
    got = steps(lines)
    assert c.get_state()["iter"] == 101
    if %d:   # steps 1..15 in a launch; 16 by itself; the launch of 17..31 is the one taken back
        assert runs(lines) == 2 and got == list(range(16, 17)) + list(range(17, 101)), lines
        assert c.timing()["step_ms"] > 0
    else:
        assert runs(lines) == 1 and got == list(range(1, 101)), lines
    c.step(50)         # the context stays on single launches
    lines = log()
    assert runs(lines) == 0 and steps(lines) == list(range(101, 151))
    """ % (stride, stride, 2 if stride else 1, stride))


def test_a_failed_launch_leaves_no_state_to_read(stub):
    """A workgroup that did not answer in time left the state half written:
    the context refuses everything but its end."""
    stub("""
    c = ocean(2)
    st = c.get_state()
    S.stub_end_resident(2, 0xffffffff)
    c.step(50)
    c.step(50, sync=False)
    assert refused(c.sync) == -2
    for call in (c.sync, c.get_state, c.dissipation, lambda: c.step(1), lambda: c.step(50),
                 lambda: c.step(1, sync=False), lambda: c.step(50, sync=False), lambda: c.velocity_en(),
                 lambda: c.dissipation_series(0, 0, 10), lambda: c.orbit_stats([0], [10]), lambda: c.retire([0]),
                 lambda: c.set_state(v=st["v"]), lambda: c.set_option(G.OPT_RESIDENT, 0),
                 lambda: c.set_sh(8, np.ones(9), mode=G.SH_RECUR)):
        assert refused(call) == -2
    assert b"did not answer" in G.lib().odis_last_error(c._h)
    c.close()
    """)


def test_no_memory_for_the_resident_step_leaves_single_launches(stub):
    """Its workspace is optional: a context that cannot have it is created and
    steps with a launch each; so does one that loses it in a retirement."""
    stub("""
    g = mesh()
    p = G.make_params(time_step=1.0)[0]
    def workspace(n):
        c = G.Context(g, [p] * n)
        c.step(20)
        held = S.stub_device_bytes()
        c.set_option(G.OPT_RESIDENT, 0)
        return held - S.stub_device_bytes()
    size = workspace(64)
    assert size > 1 << 20
    S.stub_fail_allocations_of(size)
    c = G.Context(g, [p] * 64)
    log()
    c.step(20)
    lines = log()
    assert runs(lines) == 0 and steps(lines, "il") + steps(lines) == list(range(20)), lines
    S.stub_fail_allocations_of(0)
    d = G.Context(g, [p] * 64)
    d.step(20)
    assert runs(log()) == 1
    S.stub_fail_allocations_of(workspace(63))
    d.retire(range(63))
    log()
    d.step(20)
    lines = log()
    assert runs(lines) == 0 and steps(lines) == list(range(20, 40))
    """)


def test_lds_limit_of_a_kernel_is_the_same_for_every_context(stub):
    """The limit belongs to the kernel, which all contexts of the process
    share: a smaller context must not lower it under a larger one."""
    stub("""
    big, small = ocean(level=6, tide=G.FULL2), ocean(level=4, tide=G.NONE)
    tiny = ocean(level=4, tide=G.FULL2, n=300)
    limits = {tuple(x.split()[1:]) for x in log() if x.startswith("attribute ")}
    assert limits and {v for _, v in limits} == {str(160 * 1024)}, limits
    """)


def test_calls_of_few_steps_after_a_run_do_not_wait(stub):
    """Asynchronous calls stay so: the first few of fewer steps than make a
    run are run resident behind it.  Only then does single launching, which
    has to know that the runs took place, take over; and a call now and then
    of some steps between single ones does not change it."""
    stub("""
    c = ocean()
    c.step(200, sync=False)
    log()
    for n in (1, 3, 2):
        c.step(n, sync=False)
    lines = log()
    assert runs(lines) == 3 and not [x for x in lines if x.startswith("wait")], lines
    c.step(1, sync=False)
    assert steps(log()) == [206]
    for _ in range(3):
        c.step(1, sync=False)
        c.step(4, sync=False)
    lines = log()
    assert runs(lines) == 0 and len(steps(lines)) == 15, lines
    c.step(100, sync=False)
    assert runs(log()) == 1
    assert c.get_state()["iter"] == 322
    c.step(0)
    """)


def test_a_batch_is_not_converted_at_every_call(stub):
    """Calls of one and of several steps in turn on a batch whose single steps
    are interleaved: its state stays in the layout it has until changing over
    pays."""
    stub("""
    c = ocean(16, level=7, precision=1)
    c.step(20)
    log()
    for _ in range(6):
        c.step(1)
        c.step(4)
    lines = log()
    assert runs(lines) == 12 and "convert" not in lines, lines
    for _ in range(5):
        c.step(1)                       # now interleaved
    lines = log()
    assert len(steps(lines, "il")) >= 1 and lines.count("convert") == 5, lines
    for _ in range(3):
        c.step(1)
        c.step(4)
    lines = log()
    assert len(steps(lines, "il")) == 15 and "convert" not in lines, lines
    c.step(100)
    lines = log()
    assert runs(lines) == 1 and lines.count("convert") == 5, lines
    assert c.get_state()["iter"] == 170
    """)


@pytest.mark.parametrize("case", ["ocean(), 1", "ocean(), 4", "ocean(16, level=7, precision=1), 8"])
def test_steps_sampled_closely_are_staged_together(stub, case):
    """With sampled steps closer than runs between them pay for, a call's
    steps are one chunk, as without the resident step."""
    stub("""
    c, stride = %s
    c.enable_timing(stride)
    log()
    c.step(64)
    lines = log()
    assert runs(lines) == 0 and len(steps(lines) + steps(lines, "il")) == 64
    assert sum("k_series" in x for x in lines) == 1, lines
    """ % case)


def test_launches_of_several_contexts_are_ordered_only_where_they_must_be(stub):
    """Launches whose workgroups fit the chip together are not ordered; one
    that does not fit waits for each launch of the group before it."""
    stub("""
    g, g4 = mesh(6), mesh(4)
    p = G.make_params(time_step=1.0)[0]

    def context(patches):
        c = G.Context(g if patches > 16 else g4, [p])
        c.set_option(G.OPT_RESIDENT, patches)
        return c

    def waits(c):
        log()
        c.step(8, sync=False)
        return sum(x == "after another launch" for x in log())
    small = [ocean() for _ in range(8)]          # 16 workgroups each
    assert [waits(c) for c in small + small] == [0] * 16
    for c in small:
        c.close()
    a, x, z, v = context(200), context(96), context(144), context(2)
    assert waits(a) == 0
    assert waits(x) == 1                         # after a
    assert waits(z) == 1                         # beside x, after a
    assert [waits(c) for c in (x, z, x)] == [0] * 3
    assert waits(a) == 2                         # after x and z
    assert waits(v) == 2                         # beside a, after x and z
    assert waits(x) == 2                         # after a and v
    assert waits(z) == 2                         # beside x
    assert waits(v) == 1                         # beside x and z, after a (its own is before it anyway)
    w = context(3)
    assert waits(w) == 2                         # after a and v's launch in a's group
    # the newest group's contexts end: what follows still waits for the group before
    assert waits(a) == 4
    a.close()
    S.stub_workgroups_per_cu(2)
    y = ocean(40)                                # more workgroups than compute units
    assert waits(y) == 4
    assert waits(x) == 1
    """)


def test_launches_side_by_side_fit_each_part_of_the_chip(stub):
    """A launch's workgroups go round the chip's eight parts: one of 33 may put
    five on any of them, so seven such launches do not fit parts of 32 compute
    units, though their 231 workgroups are fewer than the 256 units."""
    stub("""
    g = mesh(6)
    p = G.make_params(time_step=1.0)[0]
    cs = [G.Context(g, [p]) for _ in range(7)]
    waits = []
    for c in cs:
        c.set_option(G.OPT_RESIDENT, 33)
        log()
        c.step(8, sync=False)
        waits.append(sum(x == "after another launch" for x in log()))
    assert waits == [0] * 6 + [6], waits
    """)


def test_a_shell_holds_no_resident_step(stub):
    """Contexts coupled through spherical harmonics never run it: those that
    will be by their surface do not set it up when created, others give it back
    when a basis is set; without a basis they run it."""
    stub("""
    def grown(call):
        before = S.stub_device_bytes()
        out = call()
        return out, S.stub_device_bytes() - before
    free, b0 = grown(lambda: ocean(8))
    lid, b1 = grown(lambda: ocean(8, surface=G.LID_MEMBR, shell_thickness=20e3))
    load, b2 = grown(lambda: ocean(8, surface=G.FREE_LOADING))
    workspace = b0 - b1
    assert workspace > 1 << 19 and b1 == b2
    # (the stub computes no basis: the call ends with an error once it has the Gram matrix)
    _, f = grown(lambda: refused(lambda: free.set_sh(8, np.ones(9), mode=G.SH_RECUR)))
    _, l = grown(lambda: refused(lambda: lid.set_sh(8, np.ones(9), mode=G.SH_RECUR)))
    assert l - f == workspace
    for c in (free, lid, load):
        c.set_sh(8, np.ones(9), mode=G.SH_OFF)
        log()
        c.step(20)
        assert runs(log()) == 1
    """)


def test_the_resident_step_in_use_can_be_read_and_tried_again(stub):
    stub("""
    c = ocean()
    assert c.option(G.OPT_RESIDENT_ACTIVE) == 16                     # 642 / 40 cells
    c.set_option(G.OPT_GRAPHS, 1)
    assert c.option(G.OPT_RESIDENT_ACTIVE) == 0
    c.set_option(G.OPT_GRAPHS, 0)
    S.stub_end_resident(1, 0)
    c.step(20)
    assert c.option(G.OPT_RESIDENT_ACTIVE) == 0 and c.option(G.OPT_RESIDENT) == 1
    S.stub_end_resident(0, 0)
    c.set_option(G.OPT_RESIDENT, 1)
    log()
    c.step(20)
    assert runs(log()) == 1 and c.option(G.OPT_RESIDENT_ACTIVE) == 16
    assert refused(lambda: c.set_option(G.OPT_RESIDENT_ACTIVE, 1)) == -1
    assert ocean(3, level=2).option(G.OPT_RESIDENT_ACTIVE) >= 1     # 42 cells: one patch
    # 163842 cells in FP64 with 7 tide fields are more than the chip's LDS holds
    assert ocean(level=8, tide=G.FULL2).option(G.OPT_RESIDENT_ACTIVE) == 0
    """)


def test_a_stop_does_not_end_steps_already_taken(stub):
    """Steps accepted before a stop was requested are stepped again when their
    launch was taken back; the stop ends the next call."""
    stub("""
    c = ocean()
    S.stub_end_resident(1, 0)
    c.step(50, sync=False)
    G.lib().odis_request_stop(c._h)
    assert c.get_state()["iter"] == 50
    assert refused(lambda: c.step(10)) == -7
    c.step(10)
    assert c.get_state()["iter"] == 60
    """)


def test_cells_without_a_place_step_singly(stub):
    """Cell coordinates only order the cells and their patches; a descriptor
    whose coordinates are no numbers is still a mesh, but has no patches (NaN
    has no place in the order that cuts them)."""
    stub("""
    g = mesh()
    d = g.describe()
    lat = np.ctypeslib.as_array(ctypes.cast(d.cell_lat, ctypes.POINTER(ctypes.c_double)), (g.N,)).copy()
    lat[::3] = np.nan
    d.cell_lat = type(d.cell_lat)(lat.ctypes.data) if not hasattr(d.cell_lat, "contents") else \\
        lat.ctypes.data_as(type(d.cell_lat))
    g.describe = lambda: d
    c = G.Context(g, G.make_params(time_step=1.0)[0])
    assert c.option(G.OPT_RESIDENT_ACTIVE) == 0
    log()
    c.step(20)
    assert steps(log()) == list(range(20))
    """)
