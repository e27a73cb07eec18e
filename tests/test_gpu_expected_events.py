"""Who applies a step's nucleations is decided from a sample of the stored
energies: with none in the sampled grains and many in the others, and the other
way round, the oracle's bits."""
import numpy as np
import pytest

import sevc
from _util import Oracle, diff_fields

pytestmark = pytest.mark.gpu


# every second grain of a head that draws itself; every second, and every third,
# of a launch of its own
@pytest.mark.parametrize("n", [6_827, 8_192, 12_289])
@pytest.mark.parametrize("sampled", [0.0, 1.0])
def test_sample_that_misleads(n, sampled):
    pos, rid = sevc.voronoi(n, 6)
    rng = np.random.default_rng(6)
    o = sevc.default_options()
    o.GB_eps, o.n_grains, o.extra_capacity, o.max_vrt_per_grn, o.seed = 0.0, n, 0.2, 64, 6
    o.adaptive_dt, o.dt = 0, 1e-3 / np.sqrt(n)
    o.do_nucleation, o.nucleation_mode, o.nucleation_rate, o.nucleation_gap = 1, sevc.NUCL_RATE, 4e-3, 1
    mesh = sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)
    se = np.full(mesh.ng, 1.0 - sampled)
    se[::mesh.ng // 4096] = sampled
    assert mesh.ng // 4096 >= 2
    mesh["g_SE"][:] = 0.0
    st = sevc.State(o, mesh)
    st.set_params(0, g_SE=se)
    mesh["g_SE"][:] = se
    orc = Oracle(o, mesh)
    a, (rc, b) = st.step(6), orc.step(6)
    assert rc == 0 and a.n_nucleations == b.n_nucleations
    assert b.n_nucleations > 6 * 8
    assert diff_fields(st.get_mesh(), orc.get_mesh()) == {}
    st.close()
