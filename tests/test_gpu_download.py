"""Downloads give back what was uploaded: a mesh that fits one staged round,
one that does not (each array on its own), and lists held at another stride
than the member's, in one round and in several."""
import numpy as np
import pytest

import sevc
from sevc._abi import MESH_ARRAYS

pytestmark = pytest.mark.gpu


def _mesh(n, stride, seed):
    pos, rid = sevc.voronoi(n, seed)
    rng = np.random.default_rng(seed)
    o = sevc.default_options()
    o.n_grains, o.max_vrt_per_grn, o.extra_capacity = n, stride, 0.01
    m = sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n)
    for k in ("vel", "v_energy", "v_vel_parts", "b_energy", "b_arclength", "b_t_ext", "g_area", "g_dAdt"):
        m[k][:] = rng.random(m[k].size)
    m["b_candidate"][:] = rng.integers(0, 2, m.ne)
    m["g_type"][:] = rng.integers(0, 2, m.ng)
    return o, m


@pytest.mark.parametrize("sizes", [((12, 32), (301, 30)), ((70_001, 100), (13, 128)), ((90_000, 32),)])
def test_download(sizes):
    parts = [_mesh(n, S, 3 + k) for k, (n, S) in enumerate(sizes)]
    st = sevc.State([o for o, _ in parts], [m for _, m in parts])
    for k, (_, m) in enumerate(parts):
        got = st.get_mesh(k)
        for name, *_ in MESH_ARRAYS:
            assert np.array_equal(got[name], m[name]), (k, name)
    st.close()
