"""The raycast's far bound and its deferral inside probing runs against the
oracle: rays that leave the map (their later lookups are counted, not made)
and every deferral regime (few, many and very many lookups ahead)."""
import numpy as np
import pytest

from gpu_helpers import assert_raycast_equal, dev_u16, make_pair
from superscanner_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,vl,budget", [(1, 1, 0.005, 12), (72, 97, 0.005, 12), (72, 97, 0.005, 1),
                                           (264, 345, 0.002, 12), (264, 345, 0.002, 2), (473, 601, 0.002, 12),
                                           (721, 1281, 0.005, 12)])
def test_rays_past_the_map(gpu, H, W, vl, budget):
    cfg = dict(synth.PLAIN_SMALL, voxel_length=vl, truncation=4 * vl)
    cfg["intr"] = synth.scaled_intr(cfg, H, W)
    poses = [synth.pose_f32(T) for T in synth.traj_plain_small(n=12)[:3]]
    depth = synth.frames(synth.scene_plain_small(), poses, cfg, seed=3, H=H, W=W)
    g, o = make_pair(vl, cfg["truncation"], H, W, cfg["intr"], n_buckets=1 << 20, n_bricks=1 << 19)
    g.set_tuning(raycast_budget=budget)
    # before anything is inserted, then looking at the map, past its edge, away from it and from within it
    views = [poses[1], synth.pose_f32(synth.look_at((1.5, 0.2, 1.0), (0.0, 3.0, 0.6))),
             synth.pose_f32(synth.look_at((1.5, 0.2, 1.0), (4.0, 3.0, 2.0))),
             synth.pose_f32(synth.look_at((0.1, 0.1, 0.05), (1.0, 0.7, 0.0)))]
    assert_raycast_equal(g, o, views[0])
    for k, E in enumerate(poses):
        g.integrate(None, dev_u16(depth[k]), E)
        o.integrate(depth[k], E)
    for E in views:
        before = g.stats()
        r = assert_raycast_equal(g, o, E)
        after = g.stats()
        for name, want in (("ray_samples", "samples"), ("ray_probes", "probes"), ("ray_hits", "n_hit"),
                           ("ray_ub", "n_ub")):
            assert after[name] - before[name] == r["counts"][want], name
