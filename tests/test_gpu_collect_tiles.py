"""Collection with one patch a workgroup (small images) and with larger tiles,
on both sides of the line between them (1 024 8x8-pixel patches on 256 CUs) and
at sizes that leave partial patches and tiles, plain and as a batch, against
the oracle: the same bricks, sdf and weights."""
import numpy as np
import pytest

from gpu_helpers import assert_grids_equal, dev_u16, make_pair
from superscanner_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W", [(1, 1), (7, 9), (121, 161), (256, 256), (257, 256), (120, 547)])
@pytest.mark.parametrize("batch", [False, True])
def test_tiles_equal_oracle(gpu, H, W, batch):
    cfg = dict(synth.PLAIN_SMALL)
    cfg["intr"] = synth.scaled_intr(cfg, H, W)
    T = synth.traj_plain_small(n=9)[:4]
    poses = [synth.pose_f32(t) for t in T]
    depth = synth.frames(synth.scene_plain_small(), T, cfg, seed=5, H=H, W=W)
    signs = [1, 1, 1, -1]
    order = [0, 1, 2, 1]
    g, o = make_pair(cfg["voxel_length"], cfg["truncation"], H, W, cfg["intr"])
    if batch:
        g.integrate_batch([dev_u16(depth[k]) for k in order], [poses[k] for k in order], signs)
    for k, s in zip(order, signs):
        if not batch:
            (g.integrate if s > 0 else g.deIntegrate)(None, dev_u16(depth[k]), poses[k])
        o.integrate(depth[k], poses[k], s)
    g.sync()
    eg, _ = assert_grids_equal(g, o)
    assert len(eg["coords"]) or (H, W) == (1, 1)
    assert np.isfinite(eg["sdf"]).all()
