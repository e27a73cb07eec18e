"""A member's mesh replaced between steps: nothing of the old one is left (edits,
labels, candidate and two-triangle lists), the other members go on, and the
upload clears in one launch."""
import numpy as np
import pytest

import sevc
import _hip_calls
from _util import Oracle, diff_fields

pytestmark = pytest.mark.gpu


def _member(n, seed):
    pos, rid = sevc.voronoi(n, seed)
    rng = np.random.default_rng(seed)
    o = sevc.default_options()
    o.GB_eps, o.n_grains, o.extra_capacity, o.max_vrt_per_grn, o.seed = 0.0, n, 0.3, 64, seed
    o.adaptive_dt, o.dt, o.do_nucleation, o.flip_threshold = 0, 1e-5, 0, 0.8 / np.sqrt(n)
    return o, sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)


@pytest.mark.parametrize("replaced", [0, 1, 2])
def test_steps_after(replaced):
    ms = [_member(n, 3 + k) for k, n in enumerate((61, 700, 256))]
    st = sevc.State([o for o, _ in ms], [m for _, m in ms])
    orcs = [Oracle(o, m) for o, m in ms]
    for k in (9, 7):
        st.step(k)
        for orc in orcs:
            assert orc.step(k)[0] == 0
        st.set_mesh(replaced, ms[replaced][1])
        orcs[replaced] = Oracle(*ms[replaced])
    st.step(12)
    for k, orc in enumerate(orcs):
        assert orc.step(12)[0] == 0
        assert diff_fields(st.get_mesh(k), orc.get_mesh()) == {}, k
    st.close()


def test_no_clear_of_its_own(tmp_path):
    out = _hip_calls.run("""
pos, rid = sevc.voronoi(60, 1)
rng = np.random.default_rng(1)
o = sevc.default_options()
o.n_grains = 60
mesh = sevc.build_mesh(o, pos, rid, rng.random(60), rng.random(60), 60)
st = sevc.State(o, mesh)
hip.calls_clear()
st.set_mesh(0, mesh)
print(sum(kind == "M" for kind, _ in calls()))
""", tmp_path)
    assert out.split() == ["0"]
