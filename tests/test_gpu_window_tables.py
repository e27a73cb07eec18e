"""The window's topology tables at the shapes where they can go wrong,
against the oracle bit for bit: lists of more than 12 vertices (read past the
table), 3-sided grains, disabled slots, and lists whose order does not follow
the edges (the list neighbours are then searched for)."""
import numpy as np
import pytest

import sevc
from _util import Oracle, diff_fields

pytestmark = pytest.mark.gpu


def _nucleated(gb_eps):
    """A tessellation with many nuclei along its grains' rims, and spare slots."""
    n = 150
    pos, rid = sevc.voronoi(n, 8)
    rng = np.random.default_rng(8)
    o = sevc.default_options()
    o.GB_eps, o.n_grains, o.dt, o.max_vrt_per_grn, o.extra_capacity = gb_eps, n, 1e-5, 64, 3.0
    o.nucleation_mode, o.nucleation_rate, o.nucleation_scaling, o.seed = sevc.NUCL_RATE, 0.3, 0.5, 3
    mesh = sevc.build_mesh(o, pos, rid, rng.random(n), 0.5 + rng.random(n), n)
    orc = Oracle(o, mesh)
    assert orc.step(10)[0] == 0
    got = orc.get_mesh()
    live = got["g_enabled"] != 0
    assert got["g_vlen"][live].max() > 12 and got["g_vlen"][live].min() == 3 and not live.all()
    o.events, o.do_nucleation, o.velocity_model = 0, 0, sevc.VEL_ANALYTIC
    return o, got


def _shuffled(gb_eps):
    """A tessellation with some lists out of order (valid for check_data)."""
    o, mesh = _nucleated(gb_eps)
    rng = np.random.default_rng(1)
    lists = mesh.grain_lists()
    for g in np.nonzero(mesh["g_enabled"] * (mesh["g_vlen"] > 3))[0][::5]:
        n = mesh["g_vlen"][g]
        lists[g, :n] = rng.permutation(lists[g, :n])
    assert sevc.check_mesh(mesh)[0] == 0
    return o, mesh


@pytest.mark.parametrize("make", [_nucleated, _shuffled])
@pytest.mark.parametrize("gb_eps", [0.0, 0.3])
@pytest.mark.parametrize("steps,every", [(1, 0), (13, 5)])
def test_window_tables(make, gb_eps, steps, every):
    o, mesh = make(gb_eps)
    st, orc = sevc.State(o, mesh), Oracle(o, mesh)
    st.window_forward(steps, every)
    assert orc.window_forward(steps) == 0
    assert diff_fields(st.get_mesh(), orc.get_mesh(), ["pos", "vel", "g_area", "b_energy"]) == {}
    w = np.random.default_rng(2).standard_normal(2 * mesh.nv)
    (dp, ds, dgb, dmu), = st.adjoint(w)
    for a, b in zip((dp, ds, dgb, dmu), orc.adjoint(w)):
        assert np.array_equal(np.asarray(a).view(np.uint64), np.asarray(b).view(np.uint64))
    st.close()


def test_window_kept_and_recomputed():
    """A window past the limit of what is kept whole: its reverse pass, from
    checkpoints (the last segment a short one), against every step kept."""
    n, steps = 40_009, 1701                      # 16 + 1 bytes a vertex and step: 2.3 GB
    pos, rid = sevc.voronoi(n, 5)
    rng = np.random.default_rng(5)
    o = sevc.default_options()
    o.GB_eps, o.n_grains, o.dt = 0.3, n, 1e-4 / np.sqrt(n)
    o.events, o.do_nucleation, o.velocity_model = 0, 0, sevc.VEL_ANALYTIC
    mesh = sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)
    w = rng.standard_normal(2 * mesh.nv)
    out = []
    for every in (0, 100):
        st = sevc.State(o, mesh)
        st.window_forward(steps, every)
        (dp, ds, dgb, dmu), = st.adjoint(w)
        out.append([st.positions(0), dp, ds, np.array([dgb, dmu])])
        st.close()
    for a, b in zip(*out):
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("order", ["along the mesh", "shuffled"])
@pytest.mark.parametrize("n", [300, 70_000])
def test_window_vertex_order(order, n):
    """Vertices in no order: a block of 256 has up to 700 grains, and above 512
    blocks the area signs come from a launch of their own."""
    pos, rid = sevc.voronoi(n, 6)
    rng = np.random.default_rng(6)
    o = sevc.default_options()
    o.GB_eps, o.n_grains, o.dt = 0.0, n, 1e-4 / np.sqrt(n)
    o.events, o.do_nucleation, o.velocity_model = 0, 0, sevc.VEL_ANALYTIC
    mesh = sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)
    if order == "shuffled":
        new = rng.permutation(mesh.nv)           # slot of each vertex
        for k, width in (("pos", 2), ("v_bnd", 3), ("v_grn", 3), ("v_enabled", 1)):
            a = mesh[k].reshape(mesh.nv, width)
            b = a.copy()
            b[new] = a
            a[:] = b
        for k in ("b_vtx", "g_vtx"):
            a = mesh[k]
            a[a >= 0] = new[a[a >= 0]]
    assert sevc.check_mesh(mesh)[0] == 0
    st, orc = sevc.State(o, mesh), Oracle(o, mesh)
    st.window_forward(7, 3)
    assert orc.window_forward(7) == 0
    assert diff_fields(st.get_mesh(), orc.get_mesh(), ["pos", "vel", "g_area"]) == {}
    w = rng.standard_normal(2 * mesh.nv)
    (dp, ds, dgb, dmu), = st.adjoint(w)
    for a, b in zip((dp, ds, dgb, dmu), orc.adjoint(w)):
        assert np.array_equal(np.asarray(a).view(np.uint64), np.asarray(b).view(np.uint64))
    st.close()
