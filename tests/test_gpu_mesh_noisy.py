"""Marching cubes on bricks full of sign changes: depth that differs from pixel
to pixel gives neighbouring voxels random signs, so bricks own more vertices
than the emitting kernel sums normals for in LDS (512)."""
import numpy as np
import pytest

from gpu_helpers import dev_u8, dev_u16, make_pair
from superscanner_amd import synth
from test_gpu_mesh_cubes import assert_cubes_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage,color", [("f32", False), ("f16", False), ("f32", True)])
def test_bricks_with_many_vertices(gpu, storage, color):
    H, W, intr = 97, 129, (525.0, 525.0, 64.0, 48.0)
    g, _ = make_pair(0.005, 0.08, H, W, intr, storage=storage, with_color=color)
    rng = np.random.default_rng(7)
    depth = rng.choice([960, 1040], size=(H, W)).astype(np.uint16)  # 8 voxels before or behind
    rgb = dev_u8(rng.integers(0, 256, size=(H, W, 3))) if color else None
    g.integrate(rgb, dev_u16(depth), synth.pose_f32(synth.look_at((0.3, 0.2, 0.1), (0.31, 1.2, 0.12))))
    m = assert_cubes_equal(g, color=color)
    k = m["vertex_keys"]
    block = np.stack([((k >> s) & 0x7FFFF) >> 3 for s in (43, 24, 5)], 1)
    assert np.unique(block, axis=0, return_counts=True)[1].max() > 512
