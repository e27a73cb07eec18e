"""A refused allocation, each one of a call in turn: the call reports it, and
the same call works once there is room."""
import pytest

import _hip_calls

pytestmark = pytest.mark.gpu

START = """
pos, rid = sevc.voronoi(60, 1)
rng = np.random.default_rng(1)
o = sevc.default_options()
o.n_grains, o.GB_eps, o.dt, o.extra_capacity = 60, 0.3, 1e-5, 0.2
mesh = sevc.build_mesh(o, pos, rid, rng.random(60), rng.random(60), 60)
ranges, targets = [(0.0, 0.05, 0.005)], np.full((1, 20), 0.04)

def window():
    st = sevc.State(o, mesh)
    st.window_forward(3)
    return st

def refused(call):
    try:
        call()
    except sevc.SevcError as e:
        assert e.code == sevc.E_NOMEM, e
    else:
        raise AssertionError("not refused")
"""


def test_histogram(tmp_path):
    out = _hip_calls.run(START + """
st = window()
want = st.area_histogram(20, ranges, targets, want_grad=True)
n = 0
while True:
    st = window()
    hip.calls_refuse(n + 1, 0)
    if n == 9:
        st.area_histogram(20, ranges, targets)
        assert hip.calls_refuse_left() > 0        # no allocation is left to refuse
        break
    refused(lambda: st.area_histogram(20, ranges, targets))
    got = st.area_histogram(20, ranges, targets, want_grad=True)
    assert np.array_equal(got[0], want[0]) and got[1] == want[1] and np.array_equal(got[2][0], want[2][0])
    n += 1
print(n)
""", tmp_path)
    assert out.split() == ["9"]


def test_download(tmp_path):
    """A download needs no room of its own: without the staging (device or
    pinned memory refused, once or every time), each array goes straight; lists
    at the member's stride and at another one."""
    out = _hip_calls.run(START + """
from sevc._abi import MESH_ARRAYS
o2 = o.copy()
o2.max_vrt_per_grn = o.max_vrt_per_grn + 9
wide = sevc.build_mesh(o2, pos, rid, rng.random(60), rng.random(60), 60)
for first, more in ((1, 0), (2, 0), (1, 1000), (2, 1000)):
    for k, m in enumerate((mesh, wide)):
        st = sevc.State([o, o2], [mesh, wide])
        hip.calls_refuse(first, more)
        got = st.get_mesh(k)
        assert hip.calls_refuse_left() == (more > 0)
        hip.calls_refuse(0, 0)
        again = st.get_mesh(k)
        for name, *_ in MESH_ARRAYS:
            assert np.array_equal(got[name], again[name]), (first, more, k, name)
        for name in ("pos", "v_bnd", "v_grn", "b_vtx", "g_vtx", "g_vlen", "g_SE"):
            assert np.array_equal(got[name], m[name]), (first, more, k, name)
        st.close()
print("ok")
""", tmp_path)
    assert out.split() == ["ok"]


def test_window(tmp_path):
    """Of a window's arrays only the lists by table block (four, the last ones)
    can be done without."""
    out = _hip_calls.run(START + """
def results(st):
    st.window_forward(3)
    return [np.concatenate([np.ravel(x) for x in st.adjoint(np.arange(2.0 * mesh.nv))[0]]), st.positions(0),
            st.get_mesh()["g_area"]]

want = results(sevc.State(o, mesh))
said = []
while True:
    st = sevc.State(o, mesh)
    hip.calls_refuse(len(said) + 1, 0)
    try:
        st.window_forward(3)
        said.append("done")
    except sevc.SevcError as e:
        assert e.code == sevc.E_NOMEM
        said.append("refused")
    if hip.calls_refuse_left() > 0:                # more than the call asks for
        break
    st = sevc.State(o, mesh)
    hip.calls_refuse(len(said), 0)
    try:
        got = results(st)
    except sevc.SevcError as e:
        got = results(st)
    for a, b in zip(got, want):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64)), len(said)
    st.close()
print(*said)
""", tmp_path)
    said = out.split()
    assert said[-5:] == ["done"] * 5 and set(said[:-5]) == {"refused"}, out
