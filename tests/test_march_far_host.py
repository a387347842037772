"""The raycast march's far bound, the state of the rays it defers and the rule
of the deferral, on the host (tests/cpp/march_far_host.cpp): bit for bit the
oracle's points, depth, UB flags and counts, with every deferred ray finished
from its saved state one lookup at a time."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle
from superscanner_amd import autotune, synth
from test_march_host import HIPCC, ROOT, compare

f, i, vp = C.c_float, C.c_int, C.c_void_p


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    so = tmp_path_factory.mktemp("march") / "libmarch_far_host.so"
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off",
                    "-fhip-fp32-correctly-rounded-divide-sqrt", "-o", str(so),
                    os.path.join(ROOT, "tests", "cpp", "march_far_host.cpp")], check=True, capture_output=True)
    L = C.CDLL(str(so))
    L.march_far_host.argtypes = [i, i, f, f, f, f, f, f, f, i, vp, vp, vp, vp, C.c_uint32, vp, i, vp, vp, vp, vp]
    L.budget_of.argtypes = [i, i, i, i, i]
    return L


@pytest.fixture(scope="module", params=["plain", "room"])
def scene(request):
    if request.param == "plain":
        H, W, cfg = 97, 131, synth.PLAIN_SMALL
        poses = synth.traj_plain_small(n=12)[:4]
        views = [poses[1], synth.look_at((1.5, 0.2, 1.0), (0.0, 3.0, 0.6)), synth.look_at((1.5, 0.2, 1.0), (4.0, 3.0, 2.0)),
                 synth.look_at((0.1, 0.1, 0.05), (1.0, 0.7, 0.0))]  # at the map, past its edge, away, from within
        prims = synth.scene_plain_small()
    else:
        H, W, cfg = 73, 129, synth.ROOM_LARGE
        poses = synth.traj_random_walk(n=6, seed=2)
        views = [poses[5], poses[0]]
        prims = synth.scene_room(seed=1)
    intr = synth.scaled_intr(cfg, H, W)
    depth = synth.frames(prims, poses, dict(cfg, intr=intr), seed=3, H=H, W=W)
    o = oracle.OracleGrid(cfg["voxel_length"], cfg["truncation"], H, W)
    o.set_intrinsics(*intr)
    for d, T in zip(depth, poses):
        o.integrate(d, synth.pose_f32(T))
    return o, cfg, intr, [synth.pose_f32(T) for T in views], H, W


def raycasts(lib, o, cfg, intr, views, H, W, budget, dmax=10.0):
    """Compares every view's march with the oracle's; returns the summed counts."""
    ex = o.export()
    n = len(ex["keys"])
    nb = 1 << max(10, (2 * n).bit_length())
    total = np.zeros(8, np.uint64)
    for E in views:
        E = np.ascontiguousarray(E, np.float32).reshape(16)
        pts, dep, ub = np.zeros((H, W, 3), np.float32), np.zeros((H, W), np.float32), np.zeros((H, W), np.uint8)
        c = np.zeros(8, np.uint64)
        assert lib.march_far_host(H, W, f(intr[0]), f(intr[1]), f(intr[2]), f(intr[3]), f(cfg["voxel_length"]),
                                  f(cfg["truncation"]), f(dmax), n, ex["keys"].ctypes.data, ex["coords"].ctypes.data,
                                  ex["sdf"].ctypes.data, ex["w"].ctypes.data, C.c_uint32(nb), E.ctypes.data, budget,
                                  pts.ctypes.data, dep.ctypes.data, ub.ctypes.data, c.ctypes.data) == 0
        compare((pts, dep, ub, int(c[0]), int(c[1])), o.raycast(E.reshape(4, 4)))
        total += c
    return total


@pytest.mark.parametrize("budget", [0, 1, 2, 5, 12])
def test_far_bound_and_deferred_state(lib, scene, budget):
    o, cfg, intr, views, H, W = scene
    total = raycasts(lib, o, cfg, intr, views, H, W, budget)
    # the far bound saves lookups where rays leave the map (none do in the room's first frames)
    assert total[2] < total[3] or (cfg is synth.ROOM_LARGE and total[2] == total[3])
    deferred, in_skip, in_advance, ahead = (int(x) for x in total[4:8])
    assert (deferred > 0) == (budget > 0)
    print(f"budget {budget}: {deferred} deferred, {in_skip} in a skip, {in_advance} in a re-advance, "
          f"{ahead} with a lookup ahead")
    if cfg is synth.PLAIN_SMALL and 0 < budget < 5:
        assert in_skip and in_advance and ahead  # every kind of state


@pytest.mark.parametrize("budget", [1, 2, 3, 5])
@pytest.mark.parametrize("blocks", [1.125, 1.5])
def test_truncation_beyond_the_block(lib, blocks, budget):
    """With d_trunc > vbl the step back before a re-advance goes forward, past
    d_max where a ray hits its first block just before it: the re-advance still
    makes (and counts) its first lookup, and such a ray is not deferred."""
    H, W = 97, 131
    cfg = dict(synth.PLAIN_SMALL, voxel_length=0.01, truncation=0.08 * blocks)
    intr = synth.scaled_intr(cfg, H, W)
    poses = synth.traj_plain_small(n=12)[:3]
    depth = synth.frames(synth.scene_plain_small(), poses, dict(cfg, intr=intr), seed=3, H=H, W=W)
    for dmax in (1.0, 1.2, 1.5, 1.8):
        o = oracle.OracleGrid(cfg["voxel_length"], cfg["truncation"], H, W, max_ray_length=dmax)
        o.set_intrinsics(*intr)
        for d, T in zip(depth, poses):
            o.integrate(d, synth.pose_f32(T))
        assert raycasts(lib, o, cfg, intr, [synth.pose_f32(T) for T in poses], H, W, budget, dmax)[4] > 0
        o.close()


def test_rule_of_the_budget(lib):
    """Rays are deferred below 26 wavefronts a CU with the tile bounds, below
    6.5 without; the tuner times no budget that a raycast would ignore."""
    for W, H, with_bounds, without in ((1, 1, 1, 1), (160, 120, 1, 1), (320, 328, 1, 1), (320, 337, 1, 0),
                                       (848, 480, 1, 0), (832, 504, 1, 0), (832, 513, 0, 0), (1280, 720, 0, 0),
                                       (16384, 16384, 0, 0)):
        for b in (0, 1, 12, 4096):
            assert lib.budget_of(b, 1, W, H, 256) == (b if with_bounds else 0), (W, H)
            assert lib.budget_of(b, 0, W, H, 256) == (b if without else 0), (W, H)
    assert lib.budget_of(12, 1, 848, 480, 64) == 0  # a quarter of the CUs
    rng = np.random.default_rng(0)
    for _ in range(200):
        W, H, cu = int(rng.integers(1, 1500)), int(rng.integers(1, 1500)), int(rng.integers(1, 305))
        for skip in (0, 2):
            assert autotune.defers(skip, W, H, cu) == (lib.budget_of(12, skip == 2, W, H, cu) == 12)
        assert not autotune.defers(1, W, H, cu)
