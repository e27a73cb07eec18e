"""The route a step's events take, one launch or a launch per stage, follows the
state: also where another one comes back from a checkpoint.  Either route gives
the oracle's bits."""
import numpy as np
import pytest

import sevc
import _hip_calls
from _util import Oracle, diff_fields

pytestmark = pytest.mark.gpu


def _start():
    """More than 300 listed edges a step at first, fewer than 30 after 70 steps."""
    n = 2000
    pos, rid = sevc.voronoi(n, 5)
    rng = np.random.default_rng(5)
    o = sevc.default_options()
    o.GB_eps, o.n_grains, o.extra_capacity, o.max_vrt_per_grn, o.seed = 0.0, n, 0.3, 64, 5
    o.adaptive_dt, o.dt, o.do_nucleation, o.flip_threshold = 0, 1e-5, 0, 0.7 / np.sqrt(n)
    return o, sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)


def _routes(st, k):
    """The steps of each route among the next k."""
    st.enable_timing(True)
    before = st.kernel_times()
    st.step(k)
    after = st.kernel_times()
    st.enable_timing(False)
    return tuple(after.get(x, (0, 0))[1] - before.get(x, (0, 0))[1] for x in ("events", "poll"))


def _same(st, orc):
    return diff_fields(st.get_mesh(), orc.get_mesh()) == {}


def test_restored_state_takes_its_own_route():
    o, mesh = _start()
    st = sevc.State(o, mesh)
    st.checkpoint(0)                             # before any step: not known yet
    st.step(4)
    st.checkpoint(1)                             # busy
    st.step(90)
    st.checkpoint(2)                             # calm
    for _ in range(2):
        assert _routes(st, 4) == (4, 0)
        st.restore(0)
        assert _routes(st, 4) == (0, 4)
        st.restore(2)
        assert _routes(st, 4) == (4, 0)
        st.restore(1)
        assert _routes(st, 4) == (0, 4)
        st.restore(2)
    # a checkpoint that never saw its first step, restored after a calm stretch
    st.close()
    st = sevc.State(o, mesh)
    st.checkpoint(3)
    st.set_mesh(0, mesh)
    st.step(90)
    st.restore(3)
    assert _routes(st, 4) == (0, 4)
    st.close()


SPIKE = """
n = 16_000
pos, rid = sevc.voronoi(n, 5)
rng = np.random.default_rng(5)
o = sevc.default_options()
o.GB_eps, o.n_grains, o.extra_capacity, o.max_vrt_per_grn, o.seed = 0.0, n, 0.3, 64, 5
o.adaptive_dt, o.dt, o.do_nucleation, o.flip_threshold = 0, 1e-5, 0, 0.3 / np.sqrt(n)
mesh = sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)
st = sevc.State(o, mesh)
"""


def test_a_busy_first_step_alone():
    """A state that flips 170 edges in its first step and a third and fewer in
    those that follow: a launch per stage for the first two while it is new, for
    the first one after a restore."""
    space = {"sevc": sevc, "np": np}
    exec(SPIKE, space)
    st = space["st"]
    st.checkpoint(0)
    st.step(1)
    st.checkpoint(1)
    assert _routes(st, 20) == (19, 1)
    for _ in range(2):
        st.restore(0)
        assert _routes(st, 20) == (19, 1)
        st.restore(1)
        assert _routes(st, 20) == (20, 0)
    st.set_mesh(0, space["mesh"])
    assert _routes(st, 20) == (18, 2)
    st.restore(1)
    st.checkpoint(2)
    st.restore(0)
    st.checkpoint(3)
    st.step(30)
    st.restore(2)
    assert _routes(st, 20) == (20, 0)
    st.restore(3)
    assert _routes(st, 20) == (19, 1)
    st.close()


def test_a_busy_first_step_alone_by_graphs(tmp_path):
    """The same with captured steps: one kind of them, and the oracle's bits."""
    out = _hip_calls.run(SPIKE + """
from _util import Oracle, diff_fields
st.checkpoint(0)
orc = Oracle(o, mesh)
assert orc.step(17)[0] == 0
for _ in range(3):
    st.restore(0)
    hip.calls_clear()
    st.step(17, graph=True)
    runs = [x for kind, x in calls() if kind == "G"]
    print(len(runs), len(set(runs)), end=" ")
    assert diff_fields(st.get_mesh(), orc.get_mesh()) == {}
""", tmp_path)
    # 15 captured steps after two, then 16 after one
    assert out.split() == ["8", "2", "2", "1", "2", "1"], out


def test_route_at_the_line():
    """Both routes take the same time at some 170 listed edges: the state lists 250
    a step or more up to its 11th step, 128 and fewer from the 18th."""
    o, mesh = _start()
    st = sevc.State(o, mesh)
    st.step(7)
    assert _routes(st, 4) == (0, 4)
    st.step(9)
    assert _routes(st, 4) == (4, 0)
    st.close()


@pytest.mark.parametrize("graph", [False, True])
def test_same_bits_after_restores(graph):
    o, mesh = _start()
    st, orc = sevc.State(o, mesh), Oracle(o, mesh)
    st.checkpoint(0)
    st.step(70, graph=graph)
    st.checkpoint(1)
    for _ in range(2):
        st.restore(0)
        st.step(12, graph=graph)
        st.restore(1)
        st.step(12, graph=graph)
    assert orc.step(82)[0] == 0
    assert _same(st, orc)
    st.restore(0)
    st.step(20, graph=graph)
    orc = Oracle(o, mesh)
    assert orc.step(20)[0] == 0
    assert _same(st, orc)
    st.close()


START = """
n = 2000
pos, rid = sevc.voronoi(n, 5)
rng = np.random.default_rng(5)
o = sevc.default_options()
o.GB_eps, o.n_grains, o.extra_capacity, o.max_vrt_per_grn, o.seed = 0.0, n, 0.3, 64, 5
o.adaptive_dt, o.dt, o.do_nucleation, o.flip_threshold = 0, 1e-5, 0, 0.7 / np.sqrt(n)
mesh = sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)
st = sevc.State(o, mesh)
"""


def test_a_call_hears_of_the_device_in_time(tmp_path):
    """Every 32 steps an event is recorded, and the one before it has been
    waited for by then: a call is at most 64 steps ahead of the device."""
    out = _hip_calls.run(START + """
hip.calls_clear()
st.step(300)
made, waited = [], -1
for kind, event in calls():
    if kind == "R":
        print(len(made) - waited, end=" ")
        made.append(event)
    if kind == "S":
        waited = len(made) - 1 - made[::-1].index(event)
""", tmp_path)
    assert out.split() == ["1"] * 9


def test_a_call_of_graph_steps_follows_the_state(tmp_path):
    """A busy state that grows calm within one call changes from one captured
    run of steps to another, and each is captured once; the oracle's bits."""
    out = _hip_calls.run(START + """
from _util import Oracle, diff_fields
st.checkpoint(0)
orc = Oracle(o, mesh)
assert orc.step(257)[0] == 0
st.step(257, graph=True)
for _ in range(2):
    st.restore(0)
    hip.calls_clear()
    st.step(257, graph=True)
    runs = [x for kind, x in calls() if kind == "G"]
    kinds = sorted(set(runs), key=runs.index)
    print(len(kinds), runs == sorted(runs, key=kinds.index), hash(tuple(kinds)))
    assert diff_fields(st.get_mesh(), orc.get_mesh()) == {}
""", tmp_path)
    a, b = [x.split() for x in out.splitlines()]
    assert a[:2] == ["2", "True"] and a == b, out
