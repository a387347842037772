"""The differentiable render with its tile depth bounds and look-ahead gives
the bits of the plain march: the bounds are left out where a lookup might find
another block's brick (the alias certificate fails), the look-ahead where
coordinates may reach 2^20 voxels, so a map seen with and without either must
render and track alike."""
import numpy as np
import pytest
import torch

from gpu_helpers import dev_u16
from superscanner_amd import diff_render as dr
from superscanner_amd import synth
from superscanner_amd._lib import check
from superscanner_amd.voxel_grid import GPUVoxelGrid

pytestmark = pytest.mark.gpu

ALIAS = np.array([152, 951, 211])  # a lattice vector of the block key (tests/test_alias_lattice.py)


def plain_grid(storage, far=None):
    """The plain scene's map; far: also a few bricks of a wall at that block, away from every view."""
    cfg = dict(synth.PLAIN_SMALL)
    H, W = 240, 320
    cfg["intr"] = synth.scaled_intr(cfg, H, W)
    T = synth.traj_plain_small(n=10)
    depth = synth.frames(synth.scene_plain_small(), T, cfg, seed=2, H=H, W=W)
    g = GPUVoxelGrid(1 << 26, cfg["truncation"], cfg["voxel_length"], H, W, n_buckets=1 << 20, n_bricks=1 << 17,
                     storage=storage)
    g.setIntrinsic(*cfg["intr"])
    for k in range(len(T)):
        g.integrate(None, dev_u16(depth[k]), synth.pose_f32(T[k]))
    if far is not None:
        E = np.eye(4, dtype=np.float32)
        E[:3, 3] = far * 8 * cfg["voxel_length"]
        wall = np.zeros((H, W), np.uint16)
        wall[100:140, 140:180] = 500
        g.integrate(None, dev_u16(wall), E)
    g.sync()
    return g, T


def skewed(T, k):
    """T with its rotation's columns off unit length by k (a pose counts as rigid up to 1e-4 in R^T R)."""
    T = np.array(T, np.float64)
    T[:3, :3] *= 1.0 + 0.5 * k
    return T


def normal_eq(g, T, obs, intr):
    n, h, w = obs.shape
    ne = torch.zeros((n, 29), dtype=torch.float64, device=g.device)
    cam = dr.view_of(h, w, intr)
    check(g._L.tsdf_track_normal_eq(g._h, n, dr._fptr(dr._poses_f32(T)), cam, dr._ptr(obs), 0.1, dr._ptr(ne), None,
                                    dr._stream()), "tsdf_track_normal_eq")
    return ne


@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_bounds_equal_no_bounds(gpu, storage):
    with_bounds, T = plain_grid(storage)
    # far enough from the lattice vector that no view's block has the key of one of these bricks
    without, _ = plain_grid(storage, far=ALIAS + (100, -100, 150))
    hi = without.export_bricks()["coords"].cpu().numpy().max(0)
    reach = int(10.0 / (8 * synth.PLAIN_SMALL["voxel_length"]))  # blocks of the shortest ray's 10 m
    assert (hi + reach >= ALIAS + 60).all()  # the vector lies in (inserted box) - (probed box): no certificate
    views = [T[0], T[4],
             synth.look_at((1.5, 0.2, 1.0), (0.0, 3.0, 0.6)),   # past the map's edge
             synth.look_at((1.5, 0.2, 1.0), (4.0, 3.0, 2.0)),   # away from it
             synth.look_at((0.1, 0.1, 0.05), (1.0, 0.7, 0.0)),  # from within it
             synth.look_at((2.5, 0.0, 0.02), (0.0, 0.0, 0.01)),  # along the floor
             skewed(T[2], 5e-6), skewed(T[2], 5e-5)]  # with bounds, and too skewed for them
    for h, w, f in ((97, 131, 100.0), (240, 320, 250.0), (33, 57, 2000.0)):
        intr = (f, f, w / 2.0, h / 2.0)
        a, na = dr.render(with_bounds, views, h, w, intr, normals=True)
        b, nb = dr.render(without, views, h, w, intr, normals=True)
        assert (a[:2] > 0).any()
        assert torch.equal(a, b) and torch.equal(na, nb)
        obs = torch.where(a > 0, a + 0.01, 1.0)
        assert torch.equal(normal_eq(with_bounds, views, obs, intr), normal_eq(without, views, obs, intr))
    with_bounds.close()
    without.close()


@pytest.mark.parametrize("storage", ["f32", "f16"])
def test_look_ahead_equals_one_by_one(gpu, storage):
    """1 mm voxels some 700 m from the origin.  With rays of 10 m every
    coordinate is below 2^20 voxels; with rays of 1 km it may not be, and the
    march decides each step from the field before it takes the next.  Nothing
    lies beyond 10 m, so both see the same."""
    H, W, intr = 60, 80, (80.0, 80.0, 40.0, 30.0)
    at = np.array([300.0, -400.0, 500.0])
    rng = np.random.default_rng(4)
    y, x = np.mgrid[0:H, 0:W]
    depth = (400 + 20 * np.sin(x / 7.0) + 15 * np.cos(y / 5.0) + rng.integers(-2, 3, (H, W))).astype(np.uint16)
    depth[20:30, 30:50] = 330  # a step, with grazing sides
    depth[40:50, 10:20] = 0    # a hole
    out = []
    for dmax in (10.0, 1000.0):
        g = GPUVoxelGrid(1 << 25, 0.008, 0.001, H, W, n_buckets=1 << 18, n_bricks=1 << 16, storage=storage,
                         d_max=dmax)
        g.setIntrinsic(*intr)
        T = np.eye(4)
        T[:3, 3] = at
        for k in range(3):
            g.integrate(None, dev_u16(depth), synth.pose_f32(T))
        views = []
        for dx, ay in ((0.0, 0.0), (0.05, 0.1), (-0.08, -0.35)):
            V = np.eye(4)
            V[:3, :3] = dr.se3_exp([0, 0, 0, 0.1 * dx, ay, 0])[:3, :3]
            V[:3, 3] = at + (dx, 0.02, 0.01)
            assert (np.abs(at) + 1000.0 * np.abs(V[:3, 2])).max() > 2 ** 20 * 0.001  # the middle ray, and those around
            views.append(V)
        d, n = dr.render(g, views, 75, 101, (80.0, 80.0, 50.0, 37.0), normals=True)
        out.append((d.clone(), n.clone()))
        g.close()
    assert (out[0][0] > 0).float().mean() > 0.3
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


def test_views_on_two_streams(gpu):
    """Calls that overlap on two streams: each has its own bounds."""
    g, T = plain_grid("f32")
    h, w, intr = 240, 320, (250.0, 250.0, 160.0, 120.0)
    views = np.stack([T[k % len(T)] for k in range(16)])
    want = dr.render(g, views, h, w, intr)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for _ in range(4):
        got = []
        for s in streams + streams:
            with torch.cuda.stream(s):
                got.append(dr.render(g, views, h, w, intr))
        torch.cuda.synchronize()
        for d in got:
            assert torch.equal(d, want)
    g.close()
