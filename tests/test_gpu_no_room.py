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
