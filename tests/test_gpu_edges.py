"""Edge cases of the batched step against the oracle, bit for bit: ragged
scene sizes in one world (a floor alone, one body, a few, a full scene),
scenes of fixed bodies only, several position iterations, collisions off,
one substep and a longer time step, and a world of one body."""
from __future__ import annotations

import numpy as np
import pytest

from _libs import SimWorld, scenes, state_bits_equal

pytestmark = pytest.mark.gpu


def _compare(world, frames, check_every=10, **kw):
    o = SimWorld("orc", world)
    g = SimWorld("rp", world)
    done = 0
    while done < frames:
        n = min(check_every, frames - done)
        o.step(n, **kw)
        g.step(n, **kw)
        done += n
        bad = state_bits_equal(o.state(), g.state())
        assert not bad, f"{world.name}: {bad} differ after frame {done} ({kw})"
    for s in range(world.num_scenes):
        assert g.error(s) == 0, f"scene {s} error word {g.error(s):#x}"
    o.close()
    g.close()


def _ragged_world():
    """Scenes of 1, 2, 3, 6 and 17 bodies, and one of fixed bodies only."""
    w = scenes.World(name="ragged")
    for seed, (nc, ni) in enumerate(((0, 0), (1, 0), (1, 1), (3, 2), (8, 8))):
        scenes.drop_scene(w, 700 + seed, n_cubes=nc, n_icos=ni)
    cube = w.shape(scenes.cube_corners())
    scenes._floor(w)
    for k in range(4):  # fixed cubes resting on and above the floor
        w.add_body(cube, (1.0, 1.0, 1.0), (3.0 * k, 0.5 * k, 0.0), scenes.quaternion_new((0.0, 1.0, 0.0), 10.0 * k),
                   fixed=True)
    w.end_scene()
    return w


def test_ragged_scene_sizes_bit_exact():
    _compare(_ragged_world(), frames=120, check_every=30)


@pytest.mark.parametrize("kw", [{"iters": 4}, {"collisions": False}, {"substeps": 1, "dt": 1.0 / 30.0},
                                {"substeps": 7, "dt": 1.0 / 45.0}], ids=["iters4", "no_collisions", "one_substep",
                                                                        "seven_substeps"])
def test_step_parameters_bit_exact(kw):
    _compare(scenes.batched_uniform(4, first_seed=800), frames=60, check_every=20, **kw)


def test_single_body_world_bit_exact():
    w = scenes.World(name="one_body")
    cube = w.shape(scenes.cube_corners())
    w.add_body(cube, (0.7, 0.7, 0.7), (0.0, 3.0, 0.0), scenes.quaternion_new((1.0, 0.0, 0.0), 30.0),
               linear_velocity=(0.5, 0.0, -0.25), angular_velocity=(0.0, 2.0, 1.0))
    w.end_scene()
    _compare(w, frames=60, check_every=20)


def test_scene_of_fixed_bodies_stays_put():
    """A scene whose bodies are all fixed matches the oracle and never moves
    (fixed bodies are never written, pbd.cpp:702-711)."""
    w = scenes.World(name="all_fixed")
    cube = w.shape(scenes.cube_corners())
    scenes._floor(w)
    w.add_body(cube, (1.0, 1.0, 1.0), (0.0, -0.5, 0.0), scenes.quaternion_new((0.0, 1.0, 0.0), 0.0), fixed=True)
    w.end_scene()
    g = SimWorld("rp", w)
    before = g.state()
    g.step(30)
    moved = state_bits_equal(before, g.state(), fields=("position", "rotation"))
    assert not moved, f"fixed bodies changed {moved}"
    assert g.error(0) == 0
    g.close()
    _compare(w, frames=30, check_every=10)


@pytest.mark.parametrize("lanes,num_scenes", [(1, 3), (4, 3), (8, 3), (16, 3), (8, 67)])
def test_general_pairs_on_lane_groups_bit_exact(lanes, num_scenes):
    """Spheres against spheres, hulls and compounds on every lane-group width
    (one lane: the schedule of worlds without lane groups), and in concurrent
    views (64 scenes or more)."""
    world = scenes.batched_mixed(num_scenes, first_seed=11, n_spheres=4, n_cubes=2, n_dumbbells=3)
    o, g = SimWorld("orc", world), SimWorld("rp", world)
    assert g.lib.rp_world_set_narrow_group(g.h, lanes) == 0
    for f in range(90 if num_scenes < 10 else 45):
        o.step(1)
        g.step(1)
        if f % 15 == 14:
            bad = state_bits_equal(o.state(), g.state())
            assert not bad, f"frame {f}: differs in {bad}"
    assert not any(g.error(s) for s in range(num_scenes))


@pytest.mark.parametrize("mu", [0.0, 0.4, 0.97, 1.6])
def test_static_friction_bit_exact(mu):
    """Thin boxes (inertia of very different axes) tumbling onto each other at
    friction coefficients on both sides of what the bound on the generalized
    masses can decide without computing them, in one and in three iterations."""
    w = scenes.World(name="thin_boxes")
    cube = w.shape(scenes.cube_corners())
    rng = np.random.default_rng(17)
    for _ in range(3):
        scenes._floor(w, material=(mu, 0.5 * mu, 0.0))
        for k in range(7):
            q = rng.normal(size=4)
            w.add_body(cube, (0.9, 0.15, 0.4), (rng.uniform(-1.0, 1.0), 0.5 + 1.3 * k, rng.uniform(-1.0, 1.0)),
                       tuple(q / np.linalg.norm(q)), mass=1.0, material=(mu, 0.5 * mu, 0.1),
                       linear_velocity=(2.0, 0.0, 0.5))
        w.end_scene()
    for iters in (1, 3):
        _compare(w, frames=90, check_every=30, iters=iters)


@pytest.mark.parametrize("iters", [1, 2, 5])
def test_overlapping_sweeps_bit_exact(iters):
    """Scenes whose orders have periods from 2 to their whole depth (a lone
    cube, towers, a pile) beside one of more than 64 bodies, so that later
    sweeps start right behind or only after earlier ones."""
    w = scenes.World(name="periods")
    for k, n in enumerate((1, 2, 9, 66)):
        scenes.stack_scene(w, seed=k, num_cubes=n)
    scenes.drop_scene(w, 41, n_cubes=12, n_icos=10)
    _compare(w, frames=60, check_every=20, iters=iters)


@pytest.mark.parametrize("iters", [1, 2, 5])
def test_overlapping_joint_sweeps_change_nothing(iters):
    """Chains of two and of nine links on the floor: the sweeps on one wave, on
    half and quarter waves and on their own waves give the same bits, and the
    oracle's poses (joint limits: libm)."""
    w = scenes.World(name="chains")
    for k, n in enumerate((2, 9, 2, 1, 5)):
        scenes.chain_scene(w, 60 + k, length=n)
    o = SimWorld("orc", w)
    gs = []
    for lanes in (64, 32, 16):
        gs.append(SimWorld("rp", w))
        assert gs[-1].lib.rp_world_set_solve_lanes(gs[-1].h, lanes) == 0
    for f in range(20):
        # each frame from the device's state: a joint limit's last bit grows
        # some tenfold every few frames in these scenes
        o.set_state(gs[0].state())
        for g in [o] + gs:
            g.step(1, iters=iters)
        first = gs[0].state()
        for g in gs[1:]:
            assert not state_bits_equal(first, g.state()), f"frame {f}"
        assert np.allclose(o.state()["position"], first["position"], rtol=0, atol=1e-9), f"frame {f}"
    assert not any(g.error(s) for g in gs for s in range(w.num_scenes))


def test_scene_beyond_the_level_sort_lds_bit_exact():
    """1100 bodies in one scene that is solved level by level: its per-body
    levels lie in global memory, its level starts beyond a wave's lanes."""
    w = scenes.World(name="towers_1100")
    scenes._floor(w)
    cube = w.shape(scenes.cube_corners())
    for k in range(1100):  # 20 x 11 towers of five
        i, level = divmod(k, 5)
        w.add_body(cube, (1.0, 1.0, 1.0), (2.4 * (i % 20) - 24.0 + 0.02 * level, 2.01 * level, 2.4 * (i // 20) - 13.0),
                   scenes.quaternion_new((0.0, 1.0, 0.0), 3.0 * (k % 7)))
    w.end_scene()
    _compare(w, frames=24, check_every=8, iters=2)


@pytest.mark.parametrize("joints", [False, True])
@pytest.mark.parametrize("large", [False, True])
@pytest.mark.parametrize("others", [300, 800, 1100])
def test_solve_widths_bit_exact(others, large, joints):
    """The waves that serve a scene follow the number of scenes: a pile, a
    stack of 66 boxes and a chain among few and among many scenes keep their
    bits (against the oracle without joints)."""
    def world(n):
        w = scenes.World(name=f"among_{n}")
        scenes.drop_scene(w, 51, n_cubes=7, n_icos=7)
        if large:
            scenes.stack_scene(w, seed=3, num_cubes=66)
        if joints:
            scenes.chain_scene(w, 77, length=5)
        for s in range(n):
            scenes.drop_scene(w, 5000 + s, n_cubes=1, n_icos=0)
        return w

    few, many = world(0), world(others)
    g, h = SimWorld("rp", few), SimWorld("rp", many)
    o = SimWorld("orc", few)
    nb = few.num_bodies
    for f in range(3):
        for sim in (g, h, o):
            sim.step(15, iters=2)
        same = {k: v[:nb] for k, v in h.state().items()}
        assert not state_bits_equal(g.state(), same), f"after frame {15 * f + 15}"
        if not joints:
            assert not state_bits_equal(o.state(), same), f"after frame {15 * f + 15}"
    assert not any(g.error(s) for s in range(few.num_scenes))
    assert not any(h.error(s) for s in range(many.num_scenes))


def test_one_large_scene_among_many_small_ones_costs_little():
    """A scene of 66 bodies among 3000 small ones: the solve's waves per scene
    are not chosen by it alone (2.8 times the frame without it when they were)."""
    import time

    def frame_ms(extra):
        w = scenes.World(name="many")
        if extra:
            scenes.drop_scene(w, 9001, n_cubes=33, n_icos=32)
        for s in range(3000):
            scenes.drop_scene(w, s)
        g = SimWorld("rp", w)
        g.step(100)
        st, ms = g.state(), []
        for _ in range(5):
            g.set_state(st)
            t = time.perf_counter()
            g.step(10)
            ms.append(100.0 * (time.perf_counter() - t))
        return min(ms)

    alone, beside = frame_ms(False), frame_ms(True)
    print(f"{alone:.2f} ms per frame, {beside:.2f} with a scene of 66 bodies")
    assert beside <= 1.7 * alone


@pytest.mark.parametrize("bodies,lanes", [(6, 32), (30, 64)])
def test_two_scenes_per_wave_only_where_their_bodies_fit(bodies, lanes):
    """Many scenes share a wave by twos while the bodies of the waves that a CU
    holds fit its LDS; scenes of 30 bodies are faster with a wave each. The
    bits do not depend on it."""
    w = scenes.World(name="many")
    for s in range(1600):
        scenes.drop_scene(w, s % 40, n_cubes=bodies // 2, n_icos=bodies // 2)
    g = SimWorld("rp", w)
    assert g.lib.rp_world_solve_lanes(g.h) == lanes
    few = scenes.World(name="few")
    for s in range(40):
        scenes.drop_scene(few, s, n_cubes=bodies // 2, n_icos=bodies // 2)
    o = SimWorld("orc", few)
    g.step(60)
    o.step(60)
    st = g.state()
    for k in (0, 39):
        part = {n: v[k * few.num_bodies:(k + 1) * few.num_bodies] for n, v in st.items()}
        assert not state_bits_equal(o.state(), part), f"copy {k}"


# A device with 64 KiB of LDS per block, as far as the HIP runtime tells; what
# the kernels are launched with is recorded.
SMALL_LDS = r"""
#define __HIP_PLATFORM_AMD__
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
int largest = 0, refused = 0;
static void* real(const char* name) {
    void* hip = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
    if (!hip) hip = dlopen("libamdhip64.so", RTLD_LAZY);
    return dlsym(hip, name);
}
hipError_t hipDeviceGetAttribute(int* value, hipDeviceAttribute_t attr, int device) {
    hipError_t e = ((hipError_t(*)(int*, hipDeviceAttribute_t, int))real("hipDeviceGetAttribute"))(value, attr, device);
    if (attr == hipDeviceAttributeMaxSharedMemoryPerBlock) *value = 65536;
    return e;
}
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute attr, int value) {
    if (attr == hipFuncAttributeMaxDynamicSharedMemorySize && value > 65536) {
        ++refused;
        return hipErrorInvalidValue;
    }
    return ((hipError_t(*)(const void*, hipFuncAttribute, int))real("hipFuncSetAttribute"))(f, attr, value);
}
hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t stream) {
    if ((int)lds > largest) largest = (int)lds;
    return ((hipError_t(*)(const void*, dim3, dim3, void**, size_t, hipStream_t))real("hipLaunchKernel"))(
        f, grid, block, args, lds, stream);
}
"""
LARGE_SCENES_ON_SMALL_LDS = r"""
import ctypes, sys
sys.path.insert(0, sys.argv[1] + "/tests")
shim = ctypes.CDLL(sys.argv[2], ctypes.RTLD_GLOBAL)
from _libs import SimWorld, scenes, state_bits_equal
for bodies in (138, 141, 200):  # 64 KiB hold 141 records, less the block vote 139
    w = scenes.World(name="pile")
    scenes.drop_scene(w, 7, n_cubes=bodies // 2, n_icos=bodies - 1 - bodies // 2, grid=6)
    g, o = SimWorld("rp", w), SimWorld("orc", w)
    for sim in (g, o):
        sim.step(12)
    assert not state_bits_equal(o.state(), g.state()), bodies
    assert g.error(0) == 0
largest, refused = (ctypes.c_int.in_dll(shim, n).value for n in ("largest", "refused"))
assert refused == 0 and 138 * 464 <= largest <= 65536 - 1024, (refused, largest)
print("ok")
"""


def test_scenes_above_the_lds_of_a_small_device(tmp_path):
    """On a device with 64 KiB of LDS per block, scenes whose bodies do not fit
    are solved with the bodies in global memory, not refused."""
    from test_gpu_adjoint import _run_with_runtime

    _run_with_runtime(tmp_path, SMALL_LDS, LARGE_SCENES_ON_SMALL_LDS)


@pytest.mark.parametrize("off", [1e-13, 5e-10, 1e-5])
def test_static_friction_with_rotations_off_the_unit_sphere(off):
    """Rotations that are no unit quaternions by less and by more than the bound
    on the friction masses allows: the floor's, which no substep normalizes,
    and the bodies' at the frame's start."""
    w = scenes.World(name="off_unit")
    cube = w.shape(scenes.cube_corners())
    scenes._floor(w, material=(0.4, 0.2, 0.0))
    rng = np.random.default_rng(3)
    for k in range(7):
        q = rng.normal(size=4)
        w.add_body(cube, (0.9, 0.15, 0.4), (rng.uniform(-1.0, 1.0), 0.5 + 1.3 * k, rng.uniform(-1.0, 1.0)),
                   tuple(q / np.linalg.norm(q)), mass=1.0, material=(0.4, 0.2, 0.1), linear_velocity=(2.0, 0.0, 0.5))
    w.end_scene()
    o, g = SimWorld("orc", w), SimWorld("rp", w)
    for f in range(6):
        st = o.state()
        st["rotation"] = st["rotation"] * (1.0 + off)
        for sim in (o, g):
            sim.set_state(st)
            sim.step(10, iters=2)
        bad = state_bits_equal(o.state(), g.state())
        assert not bad, f"{bad} differ after frame {10 * f + 10}"
