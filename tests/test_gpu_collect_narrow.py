"""Collection with 64 x 8 and with 32 x 8 pixel tiles, on both sides of the two
lines between them (3 584 8x8-pixel patches on 256 CUs; a block 12 pixels wide
at 1 m, here a focal length of 300), against the oracle: the same bricks, sdf
and weights."""
import numpy as np
import pytest

from gpu_helpers import assert_grids_equal, dev_u16, make_pair
from superscanner_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,fx", [(448, 512, 500.0), (449, 512, 500.0), (449, 513, 300.0), (449, 513, 299.9),
                                    (481, 611, 301.0), (16, 16381, 5000.0)])
def test_tiles_equal_oracle(gpu, H, W, fx):
    cfg = dict(synth.PLAIN_SMALL)
    intr = cfg["intr"] = (fx, 500.0, W / 2.0, H / 2.0)
    T = synth.traj_plain_small(n=9)[:3]
    poses = [synth.pose_f32(t) for t in T]
    depth = synth.frames(synth.scene_plain_small(), T, cfg, seed=5, H=H, W=W)
    g, o = make_pair(cfg["voxel_length"], cfg["truncation"], H, W, intr, n_buckets=1 << 19)
    for k, s in ((0, 1), (1, 1), (2, 1), (1, -1)):
        (g.integrate if s > 0 else g.deIntegrate)(None, dev_u16(depth[k]), poses[k])
        o.integrate(depth[k], poses[k], s)
    g.sync()
    eg, _ = assert_grids_equal(g, o)
    assert len(eg["coords"]) and np.isfinite(eg["sdf"]).all()
