"""State I/O of a world: what is set is read back bit for bit, arrays left out
keep their values, on both sides of the size at which the arrays cross the bus
in one copy (about 19 000 bodies), and for a single body."""
import ctypes

import numpy as np
import pytest

from _libs import pkg, scenes

pytestmark = pytest.mark.gpu


def _bodies(n):
    w = scenes.World(name=f"bodies_{n}")
    cube = w.shape(scenes.cube_corners())
    for s in range(0, n, 50):
        for k in range(min(50, n - s)):
            w.add_body(cube, (0.5, 0.5, 0.5), (3.0 * k, 5.0, 0.0), (0.0, 0.0, 0.0, 1.0))
        w.end_scene()
    return w


@pytest.mark.parametrize("n", [1, 63, 1000, 19000, 20011])
def test_state_round_trip(n):
    gw = pkg.World(_bodies(n))
    rng = np.random.default_rng(n)
    st = scenes.alloc_state(n)
    for k, a in st.items():
        a[:] = rng.integers(0, 2, a.shape) if k == "active" else rng.normal(size=a.shape)
    st["position"][0, 0] = np.nan
    gw.set_state(st)
    got = gw.state()
    assert all(got[k].tobytes() == st[k].tobytes() for k in st)
    # some arrays only
    part = {k: (st[k] + 1 if k == "linear_velocity" else None) for k in st}
    gw.lib.rp_world_set_state(gw.h, ctypes.byref(scenes.state_struct(part)))
    read = {k: (np.zeros_like(st[k]) if k in ("linear_velocity", "active") else None) for k in st}
    gw.lib.rp_world_get_state(gw.h, ctypes.byref(scenes.state_struct(read)))
    assert np.array_equal(read["linear_velocity"], part["linear_velocity"])
    assert np.array_equal(read["active"], st["active"])
    assert gw.state()["rotation"].tobytes() == st["rotation"].tobytes()
