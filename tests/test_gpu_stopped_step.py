"""A step that an error in its nucleation stops has labelled nothing: the
boundaries it inserted are no candidates, however short they are (the reference
labels boundaries after the nucleation, main.cu:171-216)."""
import numpy as np
import pytest

import sevc

pytestmark = pytest.mark.gpu


def _start(n, seed):
    """Lists with room for one more vertex than the longest: a nucleation soon
    finds one full.  It is due every third step, so that the slots it takes have
    been labelled as disabled ones before."""
    pos, rid = sevc.voronoi(n, seed)
    rng = np.random.default_rng(seed)
    ori, se = rng.random(n), 0.5 + rng.random(n)
    o = sevc.default_options()
    o.GB_eps, o.n_grains, o.extra_capacity, o.max_vrt_per_grn, o.seed = 0.0, n, 0.5, 64, seed
    o.adaptive_dt, o.dt, o.flip_threshold = 0, 1e-6, 0.3 / np.sqrt(n)
    o.do_nucleation, o.nucleation_mode, o.nucleation_rate, o.nucleation_gap = 1, sevc.NUCL_RATE, 0.01, 3
    o.max_vrt_per_grn = int(sevc.build_mesh(o, pos, rid, ori, se, n)["g_vlen"].max()) + 1
    return o, sevc.build_mesh(o, pos, rid, ori, se, n)


MAX_T_EXT = 100000.0               # SEVC_MAX_T_EXT: a boundary that no step has looked at yet


@pytest.mark.parametrize("graph", [False, True])
def test_inserted_boundaries_are_no_candidates(graph):
    met = 0
    for seed in [1, 2, 3, 5, 8, 10]:
        o, mesh = _start(200, seed)
        st = sevc.State(o, mesh)
        with pytest.raises(sevc.SevcError) as stop:
            for _ in range(120):
                before = st.get_mesh()
                st.step(1, graph=graph)
        assert stop.value.code == sevc.E_GRAIN_FULL
        got = st.get_mesh()
        # (a stop in a later stage has labelled them)
        new = (got["b_enabled"] != 0) & (before["b_enabled"] == 0) & (got["b_t_ext"] == MAX_T_EXT)
        met += bool((new & (got["b_arclength"] < o.flip_threshold) & (got["b_arclength"] > 0)).any())
        assert not got["b_candidate"][new].any()
        st.close()
    assert met >= 3
