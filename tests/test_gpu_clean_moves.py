"""cleanMemory's moves: few and most of the bricks leave (more free ids than
survivors, and the reverse), fp32, fp16 and colour, bricks whose only weights
are in their last voxels, and the map in use afterwards."""
import numpy as np
import pytest

from gpu_helpers import assert_grids_equal, assert_raycast_equal, dev_u8, dev_u16, make_pair, sorted_export_gpu
from superscanner_amd import synth
from superscanner_amd.voxel_grid import GPUVoxelGrid

pytestmark = pytest.mark.gpu

H, W, N = 120, 160, 6


def frames(color=False):
    cfg = dict(synth.PLAIN_SMALL)
    intr = cfg["intr"] = synth.scaled_intr(cfg, H, W)
    T = synth.traj_plain_small(n=N)
    depth = synth.frames(synth.scene_plain_small(), T, cfg, seed=3, H=H, W=W)
    rgb = np.random.default_rng(3).integers(0, 256, (N, H, W, 3), dtype=np.uint8) if color else None
    return cfg, intr, [synth.pose_f32(t) for t in T], depth, rgb


@pytest.mark.parametrize("color", [False, True])
@pytest.mark.parametrize("gone", [1, N - 1])
def test_moves_equal_oracle(gpu, color, gone):
    cfg, intr, poses, depth, rgb = frames(color)
    g, o = make_pair(cfg["voxel_length"], cfg["truncation"], H, W, intr, with_color=color)
    col = (lambda k: dev_u8(rgb[k])) if color else (lambda k: None)
    host = (lambda k: rgb[k]) if color else (lambda k: None)
    for k in range(N):
        g.integrate(col(k), dev_u16(depth[k]), poses[k])
        o.integrate(depth[k], poses[k], 1, host(k))
    for k in range(gone):
        g.deIntegrate(col(k), dev_u16(depth[k]), poses[k])
        o.integrate(depth[k], poses[k], -1, host(k))
    n = g.size()
    removed = g.cleanMemory()
    assert removed == o.clean() and 0 < removed < n
    assert (removed > n - removed) == (gone == N - 1)
    assert_grids_equal(g, o, color=color)
    assert_raycast_equal(g, o, poses[N - 1], color=color)
    assert g.cleanMemory() == 0
    for k in range(gone):
        g.integrate(col(k), dev_u16(depth[k]), poses[k])
        o.integrate(depth[k], poses[k], 1, host(k))
    assert_grids_equal(g, o, color=color)
    assert_raycast_equal(g, o, poses[0], color=color)


@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_survivors_are_the_weighted_bricks(gpu, storage):
    """Against the export taken before: exactly the bricks with a weight stay,
    bit for bit; some of them have it in the last three quarters only."""
    cfg, intr, poses, depth, _ = frames()
    g = GPUVoxelGrid(1 << 26, cfg["truncation"], cfg["voxel_length"], H, W, n_buckets=1 << 16, n_bricks=1 << 15,
                     storage=storage)
    g.setIntrinsic(*intr)
    for k in range(N):
        g.integrate(None, dev_u16(depth[k]), poses[k])
    for k in range(3):
        g.deIntegrate(None, dev_u16(depth[k]), poses[k])
    before = sorted_export_gpu(g)
    keep = (before["w"] != 0).any(1)
    late = keep & ~(before["w"][:, :128] != 0).any(1)
    assert late.any() and not keep.all()
    assert g.cleanMemory() == int((~keep).sum())
    after = sorted_export_gpu(g)
    for name in ("coords", "sdf", "w"):
        a, b = np.ascontiguousarray(after[name]), np.ascontiguousarray(before[name][keep])
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), name
    g.close()
