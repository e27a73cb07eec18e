"""Candidate labels and the two-triangle search from the step's lists, against
the oracle bit for bit: dt bounds that list edges in vain (dt_safety above 1,
dt_min above the minimum), the fixed dt, edits of lists of any length, labels of disabled slots over calls of
one and several steps, and searches after a restore."""
import numpy as np
import pytest

import sevc
from _util import Oracle, diff_fields

pytestmark = pytest.mark.gpu


def _start(n, seed, **kw):
    pos, rid = sevc.voronoi(n, seed)
    rng = np.random.default_rng(seed)
    o = sevc.default_options()
    o.GB_eps, o.n_grains, o.extra_capacity, o.max_vrt_per_grn = 0.0, n, 0.3, 64
    o.dt = 0.2 / np.sqrt(n)
    o.do_nucleation, o.nucleation_mode, o.nucleation_rate, o.seed = 1, sevc.NUCL_RATE, 5e-3, seed
    for k, v in kw.items():
        setattr(o, k, v)
    return o, sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)


_MODES = {"safety 4": dict(adaptive_dt=1, dt_safety=4.0, flip_threshold=2e-4),
          "dt_min": dict(adaptive_dt=1, dt_safety=0.5, dt_min=3e-4, flip_threshold=1e-4),
          "adaptive": dict(adaptive_dt=1, dt_safety=0.5, flip_threshold=3e-3),
          "fixed": dict(adaptive_dt=0, dt=6e-4),
          # lists on both sides of the 16 entries that a group of lanes edits
          "long lists": dict(adaptive_dt=0, dt=2e-5, nucleation_rate=0.3, nucleation_scaling=0.5, extra_capacity=8.0)}


@pytest.mark.parametrize("n", [130, 1500])
@pytest.mark.parametrize("mode", list(_MODES))
@pytest.mark.parametrize("calls", [[1] * 12, [7, 1, 30, 2]])
def test_labels(n, mode, calls):
    o, mesh = _start(n, 21, **_MODES[mode])
    st, orc = sevc.State(o, mesh), Oracle(o, mesh)
    for k in calls:
        a = st.step(k)
        rc, b = orc.step(k)
        assert rc == 0 and (a.n_flips, a.n_removals, a.n_two_grain) == (b.n_flips, b.n_removals, b.n_two_grain)
        assert diff_fields(st.get_mesh(), orc.get_mesh()) == {}
    st.close()


@pytest.mark.parametrize("graph", [False, True])
def test_two_triangles_after_restore(graph):
    """A flip threshold of twice the mean edge leaves pairs of 3-sided grains;
    every few steps the run goes on from a restored state."""
    n = 8000
    o, mesh = _start(n, 21, adaptive_dt=0, dt=1e-5, do_nucleation=0, flip_threshold=1.2 / np.sqrt(n))
    st, orc = sevc.State(o, mesh), Oracle(o, mesh)
    total = 0
    for k in range(8):
        st.checkpoint(0)
        st.step(9, graph=graph)                  # run on, then take it back
        st.restore(0)
        a = st.step(7, graph=graph)
        rc, b = orc.step(7)
        assert rc == 0 and a.n_two_grain == b.n_two_grain
        total += b.n_two_grain
        assert diff_fields(st.get_mesh(), orc.get_mesh()) == {}
    assert total >= 2, total
    st.close()
