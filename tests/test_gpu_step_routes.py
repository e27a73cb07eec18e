"""The ways a step's launches can go, against the oracle bit for bit: the
analytic velocity with nucleation (areas on every step, whatever computes the
energies), and candidate lists on both sides of what the event stages hold in
LDS, few and many edits a step, with removals and two-triangle pairs."""
import numpy as np
import pytest

import sevc
from _util import Oracle, diff_fields

pytestmark = pytest.mark.gpu


def _start(n, seed, side=1.0, **kw):
    pos, rid = sevc.voronoi(n, seed)
    rng = np.random.default_rng(seed)
    o = sevc.default_options()
    o.domain_bound = side
    o.GB_eps, o.n_grains, o.extra_capacity, o.max_vrt_per_grn, o.seed = 0.0, n, 0.3, 64, seed
    for k, v in kw.items():
        setattr(o, k, v)
    return o, sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)


def _same(o, mesh, calls, graph=False):
    st, orc = sevc.State(o, mesh), Oracle(o, mesh)
    total = np.zeros(4, dtype=int)
    for k in calls:
        a = st.step(k, graph=graph)
        rc, b = orc.step(k)
        names = ("n_flips", "n_removals", "n_two_grain", "n_nucleations")
        want = np.array([getattr(b, x) for x in names])
        assert rc == 0 and [getattr(a, x) for x in names] == list(want)
        assert a.nucleated_area_pct == b.nucleated_area_pct
        assert diff_fields(st.get_mesh(), orc.get_mesh()) == {}
        total += want
    st.close()
    return total


@pytest.mark.parametrize("nucl", ["rate", "mc"])
@pytest.mark.parametrize("gb_eps", [0.0, 0.3])
@pytest.mark.parametrize("graph", [False, True])
def test_analytic_with_nucleation(nucl, gb_eps, graph):
    n = 400
    kw = dict(velocity_model=sevc.VEL_ANALYTIC, GB_eps=gb_eps, adaptive_dt=0, do_nucleation=1, nucleation_gap=1)
    if nucl == "rate":
        kw.update(nucleation_mode=sevc.NUCL_RATE, nucleation_rate=5e-3, dt=0.01 / np.sqrt(n))
        o, mesh = _start(n, 31, **kw)
    else:
        kw.update(nucleation_mode=sevc.NUCL_MC, MC_k=5.0, nucleation_gate=n, dt=0.01)
        o, mesh = _start(n, 31, side=20.0, **kw)
        mesh["g_SE"][:] = 3.0 + 6.0 * mesh["g_SE"]
    assert _same(o, mesh, [1, 12, 17], graph)[3] > 0


# candidates a step (192 fit the stages' LDS tables): below 80; below 140; 233
# to 46; 278 to 47; 841 to 212, past what one workgroup is given at first
@pytest.mark.parametrize("n,flip", [(90, 0.9), (180, 0.9), (500, 0.7), (2000, 0.5), (2000, 0.7)])
@pytest.mark.parametrize("calls", [[1] * 14, [14]])
def test_list_lengths(n, flip, calls):
    o, mesh = _start(n, 5, adaptive_dt=0, dt=1e-5, do_nucleation=0, flip_threshold=flip / np.sqrt(n))
    total = _same(o, mesh, calls)
    assert total[0] > 20 and total[1] > 3
