"""Marching cubes where block keys alias: a missing neighbour's 32-bit key may
be that of a brick elsewhere in the map.  That brick is not the neighbour: the
cells that reach into the missing block have unobserved corners (a missing unit
reads w = 0), and the brick's own vertices, triangles and normals stay its own.
Against the exact-coordinate oracle (oracle/mesh_cubes.py)."""
import numpy as np
import pytest

import oracle
from gpu_helpers import dev_u8, dev_u16
from superscanner_amd.voxel_grid import GPUVoxelGrid
from test_gpu_mesh_cubes import assert_cubes_equal

pytestmark = pytest.mark.gpu

ALIAS = np.array([1312, -80, 144])  # a lattice vector of the block key (tests/test_alias_lattice.py)
VL, TRUNC = 0.002, 0.008
VBL = 8 * VL


@pytest.mark.parametrize("step", [(2, 0, 0), (-2, 0, 0), (0, 2, 0), (0, -2, 0), (0, 0, 2), (0, 0, -2), (2, 2, 0),
                                  (-2, -2, 0)])
@pytest.mark.parametrize("storage,color", [("f32", False), ("f16", False), ("f32", True)])
def test_alias_of_a_missing_neighbour(gpu, storage, color, step):
    # pixels 100 mm apart on the wall, so each allocates an island of 2 x 2 x 2 blocks (its +-8 mm box), whose voxels
    # all lie in that pixel: observed up to the island's faces
    H = W = 8
    g = GPUVoxelGrid(1 << 24, TRUNC, VL, H, W, n_buckets=1 << 16, n_bricks=1 << 15, storage=storage, withColor=color)
    g.setIntrinsic(5.0, 5.0, 4.0, 4.0)
    depth = np.full((H, W), 500, np.uint16)
    rgb = dev_u8(np.random.default_rng(5).integers(0, 256, (H, W, 3))) if color else None
    # the islands, and the same ones a lattice vector and `step` blocks away: in keys they are neighbours
    for at in (np.zeros(3), ALIAS + np.array(step)):
        E = np.eye(4, dtype=np.float32)
        E[:3, 3] = at * VBL + 0.006
        g.integrate(rgb, dev_u16(depth), E)
    ex = g.export_bricks()
    blocks = {tuple(c) for c in ex["coords"].cpu().numpy()}
    keys = {oracle.prime_hash(*(int(x) for x in b)) for b in blocks}
    assert len(keys) == len(blocks)  # no two bricks of the map share a key
    steps = [(x, y, z) for x in (0, 1) for y in (0, 1) for z in (0, 1)][1:]
    around = {(b[0] + x, b[1] + y, b[2] + z) for b in blocks for x, y, z in steps}
    assert any(n not in blocks and oracle.prime_hash(*(int(x) for x in n)) in keys for n in around)
    m = assert_cubes_equal(g, color=color)
    assert len(m["faces"]) > 1000
    ext = m["vertices"][m["faces"]]
    assert (ext.max(1) - ext.min(1)).max() < 2 * VL  # no triangle is larger than its cell
    g.close()
