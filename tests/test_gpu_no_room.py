"""Calls for which the card has no room fail alone: what is called next works."""
import numpy as np
import pytest

import sevc

pytestmark = pytest.mark.gpu

TOO_LONG = 10**9                     # steps of a window: terabytes of positions


def _start(n=100):
    pos, rid = sevc.voronoi(n, 1)
    rng = np.random.default_rng(1)
    o = sevc.default_options()
    o.n_grains, o.GB_eps, o.dt = n, 0.0, 1e-5
    return o, sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)


@pytest.mark.parametrize("then", ["get_mesh", "checkpoint", "step", "step_graph", "window_forward", "create"])
def test_next_call_works(then):
    o, mesh = _start()
    st = sevc.State(o, mesh)
    with pytest.raises(sevc.SevcError) as e:
        st.window_forward(TOO_LONG)
    assert e.value.code == sevc.E_NOMEM
    if then == "create":
        sevc.State(o, mesh).close()
    elif then == "step_graph":
        assert st.step(3, graph=True).steps_done == 3
    elif then == "step":
        assert st.step(3).steps_done == 3
    elif then == "window_forward":
        st.window_forward(3)
    else:
        getattr(st, then)()
    st.close()


def test_no_reverse_pass_over_a_window_that_is_gone():
    """A window that finds no room gives the last one's arrays back first."""
    o, mesh = _start()
    o.events, o.do_nucleation, o.velocity_model = 0, 0, sevc.VEL_ANALYTIC
    w = np.random.default_rng(2).standard_normal(2 * mesh.nv)
    st = sevc.State(o, mesh)
    st.window_forward(5)
    with pytest.raises(sevc.SevcError) as e:
        st.window_forward(TOO_LONG)
    assert e.value.code == sevc.E_NOMEM
    with pytest.raises(sevc.SevcError) as e:
        st.adjoint(w)
    assert e.value.code == sevc.E_STATE
    st.window_forward(4)
    got = st.adjoint(w)[0]
    st.close()
    st = sevc.State(o, mesh)
    st.window_forward(5)
    st.window_forward(4)
    for a, b in zip(got, st.adjoint(w)[0]):
        assert np.array_equal(np.asarray(a).view(np.uint64), np.asarray(b).view(np.uint64))
    st.close()
