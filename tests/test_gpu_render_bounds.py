"""The differentiable render's tile depth bounds and look-ahead: a ray's depth
and normal do not depend on the image it is part of.  Windows of a large view
(other tiles, other wavefronts, other bounds, one of them beyond the size whose
tile map fits in LDS) give the same bits as the view; views that leave the map
or see nothing of it end with no surface."""
import pytest

from gpu_helpers import dev_u16, make_pair
from superscanner_amd import diff_render as dr
from superscanner_amd import synth

pytestmark = pytest.mark.gpu


def plain_map(storage="f32"):
    cfg = dict(synth.PLAIN_SMALL)
    H, W = 240, 320
    cfg["intr"] = synth.scaled_intr(cfg, H, W)
    T = synth.traj_plain_small(n=10)
    depth = synth.frames(synth.scene_plain_small(), T, cfg, seed=2, H=H, W=W)
    g, _ = make_pair(cfg["voxel_length"], cfg["truncation"], H, W, cfg["intr"], n_buckets=1 << 20, n_bricks=1 << 17,
                     storage=storage)
    for k in range(len(T)):
        g.integrate(None, dev_u16(depth[k]), synth.pose_f32(T[k]))
    g.sync()
    return g, T


@pytest.mark.parametrize("H,W,storage", [(1041, 1033, "f32"), (333, 501, "f32"), (333, 501, "f16")])
def test_windows_equal_the_view(gpu, H, W, storage):
    g, T = plain_map(storage)
    fx = 0.8 * W
    views = [T[0], synth.look_at((1.5, 0.2, 1.0), (0.0, 3.0, 0.6)), synth.look_at((0.1, 0.1, 0.05), (1.0, 0.7, 0.0))]
    ci, cj = float(H // 2), float(W // 2)  # exact in float, and so are their shifts
    full, nrm = dr.render(g, views, H, W, (fx, fx, cj, H - ci), normals=True)
    assert (full > 0).any(dim=2).any(dim=1).all()
    for i0, j0, h, w in ((0, 0, 65, 33), (H // 3, W // 4, 120, 97), (H - 17, W - 23, 17, 23), (H // 2, W // 2, 1, 1)):
        d, n = dr.render(g, views, h, w, (fx, fx, cj - j0, h - (ci - i0)), normals=True)
        win = (slice(None), slice(i0, i0 + h), slice(j0, j0 + w))
        assert (d == full[win]).all()
        assert (n == nrm[win]).all()


def test_views_of_nothing(gpu):
    g, T = plain_map()
    away = [synth.look_at((1.5, 0.2, 1.0), (4.0, 3.0, 2.0)), synth.look_at((60.0, 0.0, 1.0), (61.0, 0.0, 1.0))]
    assert (dr.render(g, away, 97, 131, (100.0, 100.0, 65.0, 48.0)) == 0).all()
    g.reset()  # and an empty map
    assert (dr.render(g, [T[0]], 97, 131, (100.0, 100.0, 65.0, 48.0)) == 0).all()
