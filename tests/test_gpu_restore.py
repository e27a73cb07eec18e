"""A checkpoint and its restore give back every array, at sizes on both sides of
a copy's 16 KB workgroups and of its 16-byte loads."""
import numpy as np
import pytest

import sevc
from sevc._abi import MESH_ARRAYS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [12, 61, 513, 1024, 9_001])
def test_restore(n):
    pos, rid = sevc.voronoi(n, 3)
    rng = np.random.default_rng(n)
    o = sevc.default_options()
    o.n_grains, o.extra_capacity, o.seed = n, 0.3, 5
    o.dt, o.adaptive_dt, o.nucleation_mode, o.nucleation_rate = 0.02 / np.sqrt(n), 0, sevc.NUCL_RATE, 1e-2
    st = sevc.State(o, sevc.build_mesh(o, pos, rid, rng.random(n), rng.random(n), n))
    st.step(3)
    st.checkpoint(1)
    kept = st.get_mesh()
    st.step(5)
    ahead = st.get_mesh()
    assert not np.array_equal(ahead["pos"], kept["pos"])
    for _ in range(2):
        st.restore(1)
        got = st.get_mesh()
        for name, *_ in MESH_ARRAYS:
            assert np.array_equal(got[name].view(np.uint8), kept[name].view(np.uint8)), name
        st.step(5)
        again = st.get_mesh()
        for name, *_ in MESH_ARRAYS:
            assert np.array_equal(again[name].view(np.uint8), ahead[name].view(np.uint8)), name
    st.close()
