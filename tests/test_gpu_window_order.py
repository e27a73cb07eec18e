"""Windows of a member whose mesh is replaced by one of another vertex order: the
steps form the area signs as a state created with that mesh does, with its bits."""
import numpy as np
import pytest

import sevc
from sevc._abi import MESH_ARRAYS

pytestmark = pytest.mark.gpu

STEPS = 7


def _ordered(n):
    pos, rid = sevc.voronoi(n, 9)
    rng = np.random.default_rng(9)
    o = sevc.default_options()
    o.GB_eps, o.n_grains, o.dt = 0.3, n, 1e-4 / np.sqrt(n)
    o.events, o.do_nucleation, o.velocity_model = 0, 0, sevc.VEL_ANALYTIC
    return o, sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)


def _shuffled(mesh):
    """The same mesh with its vertices numbered at random."""
    to = np.random.default_rng(4).permutation(mesh.nv)
    out = mesh.copy()
    at = np.argsort(to)
    for name, *_ in MESH_ARRAYS:
        a = mesh[name]
        if a.size % mesh.nv == 0 and name[:2] in ("po", "ve", "v_"):
            out[name][:] = a.reshape(mesh.nv, -1)[at].reshape(-1)
    for name in ("b_vtx", "g_vtx"):
        out[name][:] = np.where(mesh[name] >= 0, to[np.maximum(mesh[name], 0)], mesh[name])
    assert sevc.check_mesh(out)[0] == 0
    return out


def _window(st, w):
    """The launches that form area signs, and what a window and its reverse pass give."""
    st.enable_timing(True)
    st.window_forward(STEPS)
    st.positions(0)
    launches = st.kernel_times()["win_area"][1]
    st.enable_timing(False)
    out = [st.positions(0), st.get_mesh()["g_area"]]
    for dp, ds, dgb, dmu in st.adjoint([w] * st.n_members):
        out += [dp, ds, np.array([dgb, dmu])]
    return launches, out


@pytest.mark.parametrize("members", [1, 2])
def test_replaced_mesh(members):
    # more than 512 table blocks of 256 vertices in all
    o, mesh = _ordered(70_001 // members)
    other = _shuffled(mesh)
    w = np.random.default_rng(2).standard_normal(2 * mesh.nv)
    st = sevc.State([o] * members, [mesh] * members)
    n, _ = _window(st, w)
    assert n == 1                                   # of the last step alone
    for new in (other, mesh, other):
        for k in range(members):
            st.set_mesh(k, new)
        fresh = sevc.State([o] * members, [new] * members)
        got, want = _window(st, w), _window(fresh, w)
        assert got[0] == want[0] == (STEPS if new is other else 1)
        for a, b in zip(got[1], want[1]):
            assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
        fresh.close()
    st.close()
