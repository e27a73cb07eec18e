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
    hip.calls_refuse(n + 1)
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
