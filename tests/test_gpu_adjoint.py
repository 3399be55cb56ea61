"""The device adjoint (rp_adjoint.hip) against the oracle's dual-number build.

Scenes: a cube thrown onto a static tilted box (the differentiable workload).
The forward pass must match the oracle bit for bit (contact scenes), the
backward pass must recompute every substep bit for bit (no mismatches), and
the gradients of L = sum_s |x_cube(s) - target_s|^2 with respect to initial
velocity, angular velocity, mass and friction must equal the frozen-contact
forward-mode derivatives of the oracle (the same map) to rounding.
"""
import numpy as np
import pytest

from _libs import SimWorld, pkg, scenes, state_bits_equal
from test_oracle_dual import PARAMS, _libs, dual_gradients

pytestmark = pytest.mark.gpu

# dual slot -> column of the device gradient: state (x, q, v, w) or parameter
DEVICE_COLUMN = {"vx": ("s", 7), "vy": ("s", 8), "vz": ("s", 9), "wx": ("s", 10), "wz": ("s", 12),
                 "mass": ("p", 0), "mu_s": ("p", 1), "mu_d": ("p", 2)}


def _device_gradients(world, targets, frames):
    gw = pkg.World(world)
    assert gw.adjoint_forward(frames) == 0
    st = gw.state()
    dl = np.zeros((world.num_bodies, 13))
    for s in range(len(targets)):
        dl[2 * s + 1, 0:3] = 2.0 * (st["position"][2 * s + 1] - targets[s])
    gs, gp = gw.adjoint_backward(dl)
    assert gw.adjoint_mismatches() == 0, "backward recomputation differs from the forward pass"
    g = np.zeros((len(targets), len(PARAMS)))
    for slot, (name, _, _) in enumerate(PARAMS):
        kind, col = DEVICE_COLUMN[name]
        for s in range(len(targets)):
            g[s, slot] = gs[2 * s + 1, col] if kind == "s" else gp[2 * s + 1, col]
    return g, st, gw


@pytest.mark.parametrize("frames", [30, 120])
def test_adjoint_matches_frozen_dual_oracle(frames):
    _, dual = _libs()
    world, targets = scenes.ramps(12, first_seed=100)
    g_dev, st_dev, gw = _device_gradients(world, targets, frames)
    g_ref, st_ref = dual_gradients(dual, world, targets, frames, freeze=True)
    assert not state_bits_equal(st_dev, st_ref), "forward pass differs from the oracle"
    scale = np.maximum(np.abs(g_ref), 1e-6 * np.abs(g_ref).max(axis=1, keepdims=True) + 1e-12)
    rel = np.abs(g_dev - g_ref) / scale
    print(f"{frames} frames: max relative difference device adjoint vs dual oracle {rel.max():.3e}")
    assert rel.max() <= 1e-7, np.argwhere(rel > 1e-7)
    for s in range(world.num_scenes):
        assert gw.errors()[s] == 0


@pytest.mark.parametrize("frames", [30, 120])
def test_adjoint_agrees_with_central_differences_on_valid_scenes(frames):
    """The differentiable workload's horizon (120 frames) and a short one
    (30): on every scene whose gradient amplification is at most 10, the
    entries whose FP64 central differences are reproducible (h = 1e-6 and
    1e-7 agree to 1e-6) agree with them to 1e-6 (at least 99 % of them) and
    every one to 1e-5; the rest is the frozen-contact approximation (a
    perturbed run's contact points move, the frozen ones do not). The
    differences are plain: perturbed runs of the full step (contacts
    regenerated) on the device, whose forward pass matches the oracle bit for
    bit. Measured on 256 scenes at 30 frames: 202 valid, 1528 of 1529 valid
    reproducible entries within 1e-6; at 120 frames no scene is valid (the
    median amplification is 4e7)."""
    from raw_physics_amd import gradcheck

    r = gradcheck.gradient_check(pkg, 32, 700, frames)
    sm = r["summary"]
    print(f"{frames} frames: {sm}")
    assert r["recompute_mismatches"] == 0 and r["error_scenes"] == 0
    vs = r["stable"] & r["valid"][:, None]
    bad = np.argwhere(vs & (r["rel"] > 1e-5))
    assert len(bad) == 0, [(int(s), gradcheck.PARAMS[k], r["grads"][s, k], r["fd"][s, k], r["amplification"][s])
                           for s, k in bad]
    assert sm["agree_on_valid_reproducible"] >= 0.99 * sm["valid_reproducible_entries"]
    if frames == 30:  # before the tumbling impacts most scenes are valid
        assert sm["valid_scenes"] >= 16 and sm["valid_reproducible_entries"] >= 100


def test_autograd_function_matches_direct_adjoint():
    import torch
    from raw_physics_amd.autograd import ThrowRun, ThrowSetup

    world, targets = scenes.ramps(6, first_seed=200)
    frames = 40
    run = ThrowSetup(world, frames)
    dyn = run.dynamic
    v0 = torch.tensor(np.asarray(world.body_linear_velocity)[dyn], dtype=torch.float64, requires_grad=True)
    w0 = torch.tensor(np.asarray(world.body_angular_velocity)[dyn], dtype=torch.float64, requires_grad=True)
    mass = torch.tensor(np.asarray(world.body_mass)[dyn], dtype=torch.float64, requires_grad=True)
    mat = np.asarray(world.body_material)[dyn]
    mu_s = torch.tensor(mat[:, 0], dtype=torch.float64, requires_grad=True)
    mu_d = torch.tensor(mat[:, 1], dtype=torch.float64, requires_grad=True)
    x = ThrowRun.apply(v0, w0, mass, mu_s, mu_d, run)
    loss = ((x - torch.from_numpy(targets)) ** 2).sum()
    loss.backward()
    g_dev, _, _ = _device_gradients(world, targets, frames)
    cols = {name: k for k, (name, _, _) in enumerate(PARAMS)}
    assert np.allclose(v0.grad.numpy()[:, 0], g_dev[:, cols["vx"]], rtol=1e-12, atol=0)
    assert np.allclose(w0.grad.numpy()[:, 2], g_dev[:, cols["wz"]], rtol=1e-12, atol=0)
    assert np.allclose(mass.grad.numpy(), g_dev[:, cols["mass"]], rtol=1e-12, atol=0)
    assert np.allclose(mu_d.grad.numpy(), g_dev[:, cols["mu_d"]], rtol=1e-12, atol=0)


def test_adjoint_scope_is_enforced():
    world = scenes.batched_uniform(1)
    gw = pkg.World(world)
    assert gw.adjoint_forward(2) != 0  # 16 dynamic bodies in one scene


@pytest.mark.parametrize("scenes_n,memory", [(1, 1), (67, 1), (67, 30 << 20), (130, 0)])
def test_adjoint_record_segments_give_identical_gradients(scenes_n, memory):
    """A run recorded frame by frame (memory 1: one frame per segment), a few
    frames at a time, or whole: the same record, hence the same gradients bit
    for bit, with every substep reproduced; scenes on either side of the
    64-scene bound of the concurrent views."""
    world, _ = scenes.ramps(scenes_n, first_seed=40)
    rng = np.random.default_rng(5)
    dl = rng.normal(size=(world.num_bodies, 13))
    got = []
    for limit in (0, memory):
        gw = pkg.World(world)
        gw.set_adjoint_memory(limit)
        gw.set_views(1 if limit == 0 else 0)
        assert gw.adjoint_forward(17) == 0
        st = gw.state()
        gs, gp = gw.adjoint_backward(dl)
        assert gw.adjoint_mismatches() == 0
        assert not state_bits_equal(st, gw.state())
        got.append((gs, gp, gw.adjoint_amplification()))
    assert all(np.array_equal(a, b) for a, b in zip(*got))


# hipGraphLaunch that fails, without launching anything, on the call that
# FAIL_AT counts down to; loaded ahead of the library in a child process.
FAILING_LAUNCH = r"""
#include <dlfcn.h>
int fail_at = 0;
int hipGraphLaunch(void* exec, void* stream) {
    static int (*real)(void*, void*);
    if (!real) {
        void* hip = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
        if (!hip) hip = dlopen("libamdhip64.so", RTLD_LAZY);
        real = (int (*)(void*, void*))dlsym(hip, "hipGraphLaunch");
    }
    if (fail_at > 0 && --fail_at == 0) return 1;
    return real(exec, stream);
}
"""
FAILED_BACKWARD = r"""
import ctypes, sys
sys.path.insert(0, sys.argv[1] + "/tests")
shim = ctypes.CDLL(sys.argv[2], ctypes.RTLD_GLOBAL)
fail_at = ctypes.c_int.in_dll(shim, "fail_at")
import numpy as np
from _libs import pkg, scenes, state_bits_equal
world, _ = scenes.ramps(3, first_seed=40)
gw = pkg.World(world)
gw.set_adjoint_memory(170000)  # two frames of 82848 bytes per segment
start = gw.state()
dl = np.random.default_rng(5).normal(size=(world.num_bodies, 13))
assert gw.adjoint_forward(4) == 0
end = gw.state()
want = gw.adjoint_backward(dl)
gw.set_state(start)
assert gw.adjoint_forward(4) == 0  # the record holds the second segment again
fail_at.value = 2
try:
    gw.adjoint_backward(dl)
    raise SystemExit("the second launch was meant to fail")
except RuntimeError:
    pass
assert fail_at.value == 0
bad = state_bits_equal(end, gw.state())
assert not bad, f"the world is not left at the end of the run: {bad}"
got = gw.adjoint_backward(dl)
assert all(np.array_equal(a, b) for a, b in zip(got, want)), "gradients of a mixed record"
print("ok")
"""


def _run_with_runtime(tmp_path, runtime, code):
    """Runs `code` in a child process with functions of the HIP runtime replaced."""
    import subprocess
    import sys

    from _libs import ROOT

    src, so = tmp_path / "runtime.c", tmp_path / "runtime.so"
    src.write_text(runtime)
    subprocess.run(["gcc", "-shared", "-fPIC", "-I/opt/rocm/include", "-o", str(so), str(src), "-ldl"], check=True)
    r = subprocess.run([sys.executable, "-c", code, str(ROOT), str(so)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]


def test_failed_backward_pass_leaves_no_mixed_record(tmp_path):
    """A launch that fails while an earlier segment is stepped again: the world
    is left at the end of the recorded run, and the next backward pass does not
    take the partly overwritten record for the last segment's."""
    _run_with_runtime(tmp_path, FAILING_LAUNCH, FAILED_BACKWARD)


def test_mismatches_count_substeps():
    """A cube on a floor of fixed blocks whose corners meet under it, with more
    contacts than the backward pass keeps: the substeps that are not reproduced
    are counted once each, and the scene's error word says why."""
    w = scenes.World(name="many_blocks")
    cube = w.shape(scenes.cube_corners())
    for i in range(4):
        for j in range(4):
            w.add_body(cube, (0.3, 0.5, 0.3), (0.6 * i - 0.9, -0.5, 0.6 * j - 0.9),
                       scenes.quaternion_new((0.0, 1.0, 0.0), 0.0), fixed=True, material=(0.6, 0.5, 0.0))
    w.add_body(cube, (1.0, 0.5, 1.0), (0.01, 0.499, 0.02), scenes.quaternion_new((0.0, 1.0, 0.0), 3.0), mass=1.0,
               material=(0.6, 0.5, 0.0))
    w.end_scene()
    gw = pkg.World(w)
    frames, substeps = 4, 20
    assert gw.adjoint_forward(frames, substeps=substeps) == 0
    gw.adjoint_backward(np.ones((w.num_bodies, 13)))
    assert gw.errors()[0] & 0x800  # RP_ERR_SOLVER_CAPACITY
    n = gw.adjoint_mismatches()
    assert 0 < n <= frames * substeps, n


def test_smaller_adjoint_memory_frees_the_record():
    """A smaller limit takes effect from the next forward pass on: what the
    record of the run before it held beyond the limit is given back."""
    import ctypes

    hip = ctypes.CDLL("libamdhip64.so.7")  # the one the library runs on

    def free_bytes():
        n, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(n), ctypes.byref(total)) == 0
        return n.value

    world, _ = scenes.ramps(512, first_seed=40)
    gw = pkg.World(world)
    start = gw.state()
    dl = np.random.default_rng(5).normal(size=(world.num_bodies, 13))
    free, got = [], []
    # 20 substeps of 512 scenes: 14 MB per frame
    for limit in (0, 64 << 20):
        gw.set_adjoint_memory(limit)
        gw.set_state(start)
        assert gw.adjoint_forward(60) == 0
        got.append(gw.adjoint_backward(dl))
        free.append(free_bytes())
    assert all(np.array_equal(a, b) for a, b in zip(*got))
    assert free[1] - free[0] >= 600 << 20, free


# Counts the graphs that are instantiated.
COUNTING_INSTANTIATE = r"""
#include <dlfcn.h>
int instantiated = 0;
int hipGraphInstantiate(void** exec, void* graph, void** node, char* log, unsigned long size) {
    static int (*real)(void**, void*, void**, char*, unsigned long);
    if (!real) {
        void* hip = dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_NOLOAD);
        if (!hip) hip = dlopen("libamdhip64.so", RTLD_LAZY);
        real = (int (*)(void**, void*, void**, char*, unsigned long))dlsym(hip, "hipGraphInstantiate");
    }
    ++instantiated;
    return real(exec, graph, node, log, size);
}
"""
ALTERNATING = r"""
import ctypes, sys
sys.path.insert(0, sys.argv[1] + "/tests")
count = ctypes.c_int.in_dll(ctypes.CDLL(sys.argv[2], ctypes.RTLD_GLOBAL), "instantiated")
from _libs import SimWorld, pkg, scenes, state_bits_equal
world, _ = scenes.ramps(70, first_seed=40)
gw, oracle = pkg.World(world), SimWorld("orc", world)
for turn in range(4):
    gw.step(1)
    assert gw.adjoint_forward(2) == 0
    oracle.step(3)
    assert not state_bits_equal(oracle.state(), gw.state()), turn
    if turn == 0:
        first = count.value
assert first > 0 and count.value == first, (first, count.value)
gw.set_views(1)  # both frames' graphs are captured again, once
for turn in range(2):
    gw.step(1)
    assert gw.adjoint_forward(2) == 0
    oracle.step(3)
    assert not state_bits_equal(oracle.state(), gw.state()), turn
assert count.value == first + 2, (first, count.value)
print("ok")
"""


def test_alternating_steps_and_recorded_runs_capture_once(tmp_path):
    """A loop that steps and records in turn keeps both frames' graphs."""
    _run_with_runtime(tmp_path, COUNTING_INSTANTIATE, ALTERNATING)


@pytest.mark.parametrize("copies", [1, 66])
def test_record_of_scenes_with_many_fixed_bodies(copies):
    """Fixed bodies never pair with each other, so the record has a slot per
    body and not per pair of bodies (4.5 GB a frame here for one scene), in one
    view and in concurrent ones; bodies out of reach change no gradient."""
    import ctypes

    hip = ctypes.CDLL("libamdhip64.so.7")  # the one the library runs on

    def free_bytes():
        n, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(n), ctypes.byref(total)) == 0
        return n.value

    def world(far):
        w = scenes.World(name="thrown")
        cube = w.shape(scenes.cube_corners())
        for s in range(copies):
            scenes._floor(w)
            w.add_body(cube, (0.5, 0.4, 0.3), (0.0, -0.2 + 0.01 * s, 0.0), scenes.quaternion_new((0.0, 0.0, 1.0), 20.0 + s),
                       mass=1.0, material=(0.6, 0.5, 0.0), linear_velocity=(2.0, -1.0, 0.3))
            for k in range(far):
                w.add_body(cube, (0.5, 0.5, 0.5), (10.0 + 2.0 * (k % 25), 20.0, 2.0 * (k // 25)),
                           scenes.quaternion_new((0.0, 1.0, 0.0), 0.0), fixed=True)
            w.end_scene()
        return w

    out = []
    for far in (0, 550 if copies == 1 else 40):
        w = world(far)
        gw = pkg.World(w)
        dl = np.zeros((w.num_bodies, 13))
        dyn = 1 + (2 + far) * np.arange(copies)
        dl[dyn] = np.random.default_rng(1).normal(size=(copies, 13))
        before = free_bytes()
        assert gw.adjoint_forward(20) == 0
        gs, gp = gw.adjoint_backward(dl)
        assert gw.adjoint_mismatches() == 0 and not gw.errors().any()
        assert before - free_bytes() < 2 << 30
        out.append((gs[dyn], gp[dyn], gw.state()["position"][dyn]))
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    assert np.abs(out[0][1]).max() > 0.0  # (friction and mass matter: it has landed)
