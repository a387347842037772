// tsdf_mc.hpp -- marching cubes over the bricks, the mesh the reference
// builds in marchingCubesHost (GPUVoxelGrid.cpp:200-251): the bricks are
// copied into an Open3D 0.12 ScalableTSDFVolume (8^3 voxels per unit, RGB8
// colour) and meshed by its ExtractTriangleMesh (:248), then
// ComputeVertexNormals (:249).  Included once, at the end of tsdf_hip.hip.
//
// The copy at GPUVoxelGrid.cpp:226-241 walks (x, y, z) with z fastest and
// stores voxel x + 8y + 64z of the brick (storage order) at Open3D index
// x + 8y + 64z, which Open3D's UniformTSDFVolume::IndexOf reads as voxel
// (z, y, x) (its index is 64 X + 8 Y + Z); the voxel it reads there is
// storage voxel (z, y, x), so the two transpositions cancel and the volume
// holds each voxel at its own (x, y, z).  Semantics of ExtractTriangleMesh
// (Open3D's own implementation of Bourke's "Polygonising a scalar field"
// with the Lorensen-Cline case tables), restated:
//   * cell (x, y, z) of unit (bx, by, bz) has corners k = 0..7 at voxel
//     (x, y, z) + offset(k) (0,0,0) (1,0,0) (1,1,0) (0,1,0) (0,0,1) (1,0,1)
//     (1,1,1) (0,1,1), in the same unit or the next one along an axis (a
//     missing unit reads w = 0);
//   * a corner with w == 0 drops the cell (so w = -1, a deintegration
//     remainder, counts as observed); otherwise bit k of the case is
//     sdf_k < 0; cases 0 and 255 emit nothing;
//   * a vertex per lattice edge: edge (global voxel G, axis a) from G to
//     G + e_a, position (vl/2 + vl G) in double with
//     f0 vl / (f0 + f1) added along a, f0 = |sdf(G)|, f1 = |sdf(G + e_a)|
//     (doubles); colour (f1 c0 + f0 c1) / (f0 + f1) with c = rgb / 255;
//     every cell that shares the edge shares the vertex;
//   * triangle t of the case row (e[3t], e[3t+1], e[3t+2]) is emitted as
//     (e[3t], e[3t+2], e[3t+1]), which faces the positive (free-space) side;
//   * vertex normal = sum of the unnormalised face normals (v1 - v0) x
//     (v2 - v0) of its triangles, then normalised (a zero sum stays zero).
// Open3D's vertex and triangle order follows its hash-map iteration order;
// here triangles and vertices come in brick order, cells in x + 8y + 64z
// order and edges by axis, then voxel, within a brick (brick ids depend on the
// order of allocation), so the mesh equals the reference's as a set of
// vertices (each named by its edge) and a multiset of triangles over them.
#pragma once

namespace {

// Corner k's offset as bits x + 2y + 4z.
__constant__ uint8_t kMcCorner[8] = {0, 1, 3, 2, 4, 5, 7, 6};
// Edge e runs from corner kMcEdgeLo[e] to corner kMcEdgeHi[e] along axis
// kMcEdgeAxis[e] (the low corner first).
__constant__ uint8_t kMcEdgeLo[12] = {0, 1, 3, 0, 4, 5, 7, 4, 0, 1, 2, 3};
__constant__ uint8_t kMcEdgeHi[12] = {1, 2, 2, 3, 5, 6, 6, 7, 4, 5, 6, 7};
__constant__ uint8_t kMcEdgeAxis[12] = {0, 1, 0, 1, 0, 1, 0, 1, 2, 2, 2, 2};
// Triangles of each case (bit k = corner k inside), edges in threes, -1
// terminated: the published Lorensen-Cline / Bourke table.
__constant__ int8_t kMcTri[256][16] = {
    {-1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 8, 3, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 1, 9, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {1, 8, 3, 9, 8, 1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {1, 2, 10, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 8, 3, 1, 2, 10, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {9, 2, 10, 0, 2, 9, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {2, 8, 3, 2, 10, 8, 10, 9, 8, -1, -1, -1, -1, -1, -1, -1},
    {3, 11, 2, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 11, 2, 8, 11, 0, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {1, 9, 0, 2, 3, 11, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {1, 11, 2, 1, 9, 11, 9, 8, 11, -1, -1, -1, -1, -1, -1, -1},
    {3, 10, 1, 11, 10, 3, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 10, 1, 0, 8, 10, 8, 11, 10, -1, -1, -1, -1, -1, -1, -1},
    {3, 9, 0, 3, 11, 9, 11, 10, 9, -1, -1, -1, -1, -1, -1, -1},
    {9, 8, 10, 10, 8, 11, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {4, 7, 8, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {4, 3, 0, 7, 3, 4, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 1, 9, 8, 4, 7, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {4, 1, 9, 4, 7, 1, 7, 3, 1, -1, -1, -1, -1, -1, -1, -1},
    {1, 2, 10, 8, 4, 7, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {3, 4, 7, 3, 0, 4, 1, 2, 10, -1, -1, -1, -1, -1, -1, -1},
    {9, 2, 10, 9, 0, 2, 8, 4, 7, -1, -1, -1, -1, -1, -1, -1},
    {2, 10, 9, 2, 9, 7, 2, 7, 3, 7, 9, 4, -1, -1, -1, -1},
    {8, 4, 7, 3, 11, 2, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {11, 4, 7, 11, 2, 4, 2, 0, 4, -1, -1, -1, -1, -1, -1, -1},
    {9, 0, 1, 8, 4, 7, 2, 3, 11, -1, -1, -1, -1, -1, -1, -1},
    {4, 7, 11, 9, 4, 11, 9, 11, 2, 9, 2, 1, -1, -1, -1, -1},
    {3, 10, 1, 3, 11, 10, 7, 8, 4, -1, -1, -1, -1, -1, -1, -1},
    {1, 11, 10, 1, 4, 11, 1, 0, 4, 7, 11, 4, -1, -1, -1, -1},
    {4, 7, 8, 9, 0, 11, 9, 11, 10, 11, 0, 3, -1, -1, -1, -1},
    {4, 7, 11, 4, 11, 9, 9, 11, 10, -1, -1, -1, -1, -1, -1, -1},
    {9, 5, 4, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {9, 5, 4, 0, 8, 3, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 5, 4, 1, 5, 0, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {8, 5, 4, 8, 3, 5, 3, 1, 5, -1, -1, -1, -1, -1, -1, -1},
    {1, 2, 10, 9, 5, 4, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {3, 0, 8, 1, 2, 10, 4, 9, 5, -1, -1, -1, -1, -1, -1, -1},
    {5, 2, 10, 5, 4, 2, 4, 0, 2, -1, -1, -1, -1, -1, -1, -1},
    {2, 10, 5, 3, 2, 5, 3, 5, 4, 3, 4, 8, -1, -1, -1, -1},
    {9, 5, 4, 2, 3, 11, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 11, 2, 0, 8, 11, 4, 9, 5, -1, -1, -1, -1, -1, -1, -1},
    {0, 5, 4, 0, 1, 5, 2, 3, 11, -1, -1, -1, -1, -1, -1, -1},
    {2, 1, 5, 2, 5, 8, 2, 8, 11, 4, 8, 5, -1, -1, -1, -1},
    {10, 3, 11, 10, 1, 3, 9, 5, 4, -1, -1, -1, -1, -1, -1, -1},
    {4, 9, 5, 0, 8, 1, 8, 10, 1, 8, 11, 10, -1, -1, -1, -1},
    {5, 4, 0, 5, 0, 11, 5, 11, 10, 11, 0, 3, -1, -1, -1, -1},
    {5, 4, 8, 5, 8, 10, 10, 8, 11, -1, -1, -1, -1, -1, -1, -1},
    {9, 7, 8, 5, 7, 9, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {9, 3, 0, 9, 5, 3, 5, 7, 3, -1, -1, -1, -1, -1, -1, -1},
    {0, 7, 8, 0, 1, 7, 1, 5, 7, -1, -1, -1, -1, -1, -1, -1},
    {1, 5, 3, 3, 5, 7, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {9, 7, 8, 9, 5, 7, 10, 1, 2, -1, -1, -1, -1, -1, -1, -1},
    {10, 1, 2, 9, 5, 0, 5, 3, 0, 5, 7, 3, -1, -1, -1, -1},
    {8, 0, 2, 8, 2, 5, 8, 5, 7, 10, 5, 2, -1, -1, -1, -1},
    {2, 10, 5, 2, 5, 3, 3, 5, 7, -1, -1, -1, -1, -1, -1, -1},
    {7, 9, 5, 7, 8, 9, 3, 11, 2, -1, -1, -1, -1, -1, -1, -1},
    {9, 5, 7, 9, 7, 2, 9, 2, 0, 2, 7, 11, -1, -1, -1, -1},
    {2, 3, 11, 0, 1, 8, 1, 7, 8, 1, 5, 7, -1, -1, -1, -1},
    {11, 2, 1, 11, 1, 7, 7, 1, 5, -1, -1, -1, -1, -1, -1, -1},
    {9, 5, 8, 8, 5, 7, 10, 1, 3, 10, 3, 11, -1, -1, -1, -1},
    {5, 7, 0, 5, 0, 9, 7, 11, 0, 1, 0, 10, 11, 10, 0, -1},
    {11, 10, 0, 11, 0, 3, 10, 5, 0, 8, 0, 7, 5, 7, 0, -1},
    {11, 10, 5, 7, 11, 5, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {10, 6, 5, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 8, 3, 5, 10, 6, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {9, 0, 1, 5, 10, 6, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {1, 8, 3, 1, 9, 8, 5, 10, 6, -1, -1, -1, -1, -1, -1, -1},
    {1, 6, 5, 2, 6, 1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {1, 6, 5, 1, 2, 6, 3, 0, 8, -1, -1, -1, -1, -1, -1, -1},
    {9, 6, 5, 9, 0, 6, 0, 2, 6, -1, -1, -1, -1, -1, -1, -1},
    {5, 9, 8, 5, 8, 2, 5, 2, 6, 3, 2, 8, -1, -1, -1, -1},
    {2, 3, 11, 10, 6, 5, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {11, 0, 8, 11, 2, 0, 10, 6, 5, -1, -1, -1, -1, -1, -1, -1},
    {0, 1, 9, 2, 3, 11, 5, 10, 6, -1, -1, -1, -1, -1, -1, -1},
    {5, 10, 6, 1, 9, 2, 9, 11, 2, 9, 8, 11, -1, -1, -1, -1},
    {6, 3, 11, 6, 5, 3, 5, 1, 3, -1, -1, -1, -1, -1, -1, -1},
    {0, 8, 11, 0, 11, 5, 0, 5, 1, 5, 11, 6, -1, -1, -1, -1},
    {3, 11, 6, 0, 3, 6, 0, 6, 5, 0, 5, 9, -1, -1, -1, -1},
    {6, 5, 9, 6, 9, 11, 11, 9, 8, -1, -1, -1, -1, -1, -1, -1},
    {5, 10, 6, 4, 7, 8, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {4, 3, 0, 4, 7, 3, 6, 5, 10, -1, -1, -1, -1, -1, -1, -1},
    {1, 9, 0, 5, 10, 6, 8, 4, 7, -1, -1, -1, -1, -1, -1, -1},
    {10, 6, 5, 1, 9, 7, 1, 7, 3, 7, 9, 4, -1, -1, -1, -1},
    {6, 1, 2, 6, 5, 1, 4, 7, 8, -1, -1, -1, -1, -1, -1, -1},
    {1, 2, 5, 5, 2, 6, 3, 0, 4, 3, 4, 7, -1, -1, -1, -1},
    {8, 4, 7, 9, 0, 5, 0, 6, 5, 0, 2, 6, -1, -1, -1, -1},
    {7, 3, 9, 7, 9, 4, 3, 2, 9, 5, 9, 6, 2, 6, 9, -1},
    {3, 11, 2, 7, 8, 4, 10, 6, 5, -1, -1, -1, -1, -1, -1, -1},
    {5, 10, 6, 4, 7, 2, 4, 2, 0, 2, 7, 11, -1, -1, -1, -1},
    {0, 1, 9, 4, 7, 8, 2, 3, 11, 5, 10, 6, -1, -1, -1, -1},
    {9, 2, 1, 9, 11, 2, 9, 4, 11, 7, 11, 4, 5, 10, 6, -1},
    {8, 4, 7, 3, 11, 5, 3, 5, 1, 5, 11, 6, -1, -1, -1, -1},
    {5, 1, 11, 5, 11, 6, 1, 0, 11, 7, 11, 4, 0, 4, 11, -1},
    {0, 5, 9, 0, 6, 5, 0, 3, 6, 11, 6, 3, 8, 4, 7, -1},
    {6, 5, 9, 6, 9, 11, 4, 7, 9, 7, 11, 9, -1, -1, -1, -1},
    {10, 4, 9, 6, 4, 10, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {4, 10, 6, 4, 9, 10, 0, 8, 3, -1, -1, -1, -1, -1, -1, -1},
    {10, 0, 1, 10, 6, 0, 6, 4, 0, -1, -1, -1, -1, -1, -1, -1},
    {8, 3, 1, 8, 1, 6, 8, 6, 4, 6, 1, 10, -1, -1, -1, -1},
    {1, 4, 9, 1, 2, 4, 2, 6, 4, -1, -1, -1, -1, -1, -1, -1},
    {3, 0, 8, 1, 2, 9, 2, 4, 9, 2, 6, 4, -1, -1, -1, -1},
    {0, 2, 4, 4, 2, 6, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {8, 3, 2, 8, 2, 4, 4, 2, 6, -1, -1, -1, -1, -1, -1, -1},
    {10, 4, 9, 10, 6, 4, 11, 2, 3, -1, -1, -1, -1, -1, -1, -1},
    {0, 8, 2, 2, 8, 11, 4, 9, 10, 4, 10, 6, -1, -1, -1, -1},
    {3, 11, 2, 0, 1, 6, 0, 6, 4, 6, 1, 10, -1, -1, -1, -1},
    {6, 4, 1, 6, 1, 10, 4, 8, 1, 2, 1, 11, 8, 11, 1, -1},
    {9, 6, 4, 9, 3, 6, 9, 1, 3, 11, 6, 3, -1, -1, -1, -1},
    {8, 11, 1, 8, 1, 0, 11, 6, 1, 9, 1, 4, 6, 4, 1, -1},
    {3, 11, 6, 3, 6, 0, 0, 6, 4, -1, -1, -1, -1, -1, -1, -1},
    {6, 4, 8, 11, 6, 8, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {7, 10, 6, 7, 8, 10, 8, 9, 10, -1, -1, -1, -1, -1, -1, -1},
    {0, 7, 3, 0, 10, 7, 0, 9, 10, 6, 7, 10, -1, -1, -1, -1},
    {10, 6, 7, 1, 10, 7, 1, 7, 8, 1, 8, 0, -1, -1, -1, -1},
    {10, 6, 7, 10, 7, 1, 1, 7, 3, -1, -1, -1, -1, -1, -1, -1},
    {1, 2, 6, 1, 6, 8, 1, 8, 9, 8, 6, 7, -1, -1, -1, -1},
    {2, 6, 9, 2, 9, 1, 6, 7, 9, 0, 9, 3, 7, 3, 9, -1},
    {7, 8, 0, 7, 0, 6, 6, 0, 2, -1, -1, -1, -1, -1, -1, -1},
    {7, 3, 2, 6, 7, 2, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {2, 3, 11, 10, 6, 8, 10, 8, 9, 8, 6, 7, -1, -1, -1, -1},
    {2, 0, 7, 2, 7, 11, 0, 9, 7, 6, 7, 10, 9, 10, 7, -1},
    {1, 8, 0, 1, 7, 8, 1, 10, 7, 6, 7, 10, 2, 3, 11, -1},
    {11, 2, 1, 11, 1, 7, 10, 6, 1, 6, 7, 1, -1, -1, -1, -1},
    {8, 9, 6, 8, 6, 7, 9, 1, 6, 11, 6, 3, 1, 3, 6, -1},
    {0, 9, 1, 11, 6, 7, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {7, 8, 0, 7, 0, 6, 3, 11, 0, 11, 6, 0, -1, -1, -1, -1},
    {7, 11, 6, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {7, 6, 11, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {3, 0, 8, 11, 7, 6, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 1, 9, 11, 7, 6, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {8, 1, 9, 8, 3, 1, 11, 7, 6, -1, -1, -1, -1, -1, -1, -1},
    {10, 1, 2, 6, 11, 7, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {1, 2, 10, 3, 0, 8, 6, 11, 7, -1, -1, -1, -1, -1, -1, -1},
    {2, 9, 0, 2, 10, 9, 6, 11, 7, -1, -1, -1, -1, -1, -1, -1},
    {6, 11, 7, 2, 10, 3, 10, 8, 3, 10, 9, 8, -1, -1, -1, -1},
    {7, 2, 3, 6, 2, 7, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {7, 0, 8, 7, 6, 0, 6, 2, 0, -1, -1, -1, -1, -1, -1, -1},
    {2, 7, 6, 2, 3, 7, 0, 1, 9, -1, -1, -1, -1, -1, -1, -1},
    {1, 6, 2, 1, 8, 6, 1, 9, 8, 8, 7, 6, -1, -1, -1, -1},
    {10, 7, 6, 10, 1, 7, 1, 3, 7, -1, -1, -1, -1, -1, -1, -1},
    {10, 7, 6, 1, 7, 10, 1, 8, 7, 1, 0, 8, -1, -1, -1, -1},
    {0, 3, 7, 0, 7, 10, 0, 10, 9, 6, 10, 7, -1, -1, -1, -1},
    {7, 6, 10, 7, 10, 8, 8, 10, 9, -1, -1, -1, -1, -1, -1, -1},
    {6, 8, 4, 11, 8, 6, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {3, 6, 11, 3, 0, 6, 0, 4, 6, -1, -1, -1, -1, -1, -1, -1},
    {8, 6, 11, 8, 4, 6, 9, 0, 1, -1, -1, -1, -1, -1, -1, -1},
    {9, 4, 6, 9, 6, 3, 9, 3, 1, 11, 3, 6, -1, -1, -1, -1},
    {6, 8, 4, 6, 11, 8, 2, 10, 1, -1, -1, -1, -1, -1, -1, -1},
    {1, 2, 10, 3, 0, 11, 0, 6, 11, 0, 4, 6, -1, -1, -1, -1},
    {4, 11, 8, 4, 6, 11, 0, 2, 9, 2, 10, 9, -1, -1, -1, -1},
    {10, 9, 3, 10, 3, 2, 9, 4, 3, 11, 3, 6, 4, 6, 3, -1},
    {8, 2, 3, 8, 4, 2, 4, 6, 2, -1, -1, -1, -1, -1, -1, -1},
    {0, 4, 2, 4, 6, 2, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {1, 9, 0, 2, 3, 4, 2, 4, 6, 4, 3, 8, -1, -1, -1, -1},
    {1, 9, 4, 1, 4, 2, 2, 4, 6, -1, -1, -1, -1, -1, -1, -1},
    {8, 1, 3, 8, 6, 1, 8, 4, 6, 6, 10, 1, -1, -1, -1, -1},
    {10, 1, 0, 10, 0, 6, 6, 0, 4, -1, -1, -1, -1, -1, -1, -1},
    {4, 6, 3, 4, 3, 8, 6, 10, 3, 0, 3, 9, 10, 9, 3, -1},
    {10, 9, 4, 6, 10, 4, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {4, 9, 5, 7, 6, 11, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 8, 3, 4, 9, 5, 11, 7, 6, -1, -1, -1, -1, -1, -1, -1},
    {5, 0, 1, 5, 4, 0, 7, 6, 11, -1, -1, -1, -1, -1, -1, -1},
    {11, 7, 6, 8, 3, 4, 3, 5, 4, 3, 1, 5, -1, -1, -1, -1},
    {9, 5, 4, 10, 1, 2, 7, 6, 11, -1, -1, -1, -1, -1, -1, -1},
    {6, 11, 7, 1, 2, 10, 0, 8, 3, 4, 9, 5, -1, -1, -1, -1},
    {7, 6, 11, 5, 4, 10, 4, 2, 10, 4, 0, 2, -1, -1, -1, -1},
    {3, 4, 8, 3, 5, 4, 3, 2, 5, 10, 5, 2, 11, 7, 6, -1},
    {7, 2, 3, 7, 6, 2, 5, 4, 9, -1, -1, -1, -1, -1, -1, -1},
    {9, 5, 4, 0, 8, 6, 0, 6, 2, 6, 8, 7, -1, -1, -1, -1},
    {3, 6, 2, 3, 7, 6, 1, 5, 0, 5, 4, 0, -1, -1, -1, -1},
    {6, 2, 8, 6, 8, 7, 2, 1, 8, 4, 8, 5, 1, 5, 8, -1},
    {9, 5, 4, 10, 1, 6, 1, 7, 6, 1, 3, 7, -1, -1, -1, -1},
    {1, 6, 10, 1, 7, 6, 1, 0, 7, 8, 7, 0, 9, 5, 4, -1},
    {4, 0, 10, 4, 10, 5, 0, 3, 10, 6, 10, 7, 3, 7, 10, -1},
    {7, 6, 10, 7, 10, 8, 5, 4, 10, 4, 8, 10, -1, -1, -1, -1},
    {6, 9, 5, 6, 11, 9, 11, 8, 9, -1, -1, -1, -1, -1, -1, -1},
    {3, 6, 11, 0, 6, 3, 0, 5, 6, 0, 9, 5, -1, -1, -1, -1},
    {0, 11, 8, 0, 5, 11, 0, 1, 5, 5, 6, 11, -1, -1, -1, -1},
    {6, 11, 3, 6, 3, 5, 5, 3, 1, -1, -1, -1, -1, -1, -1, -1},
    {1, 2, 10, 9, 5, 11, 9, 11, 8, 11, 5, 6, -1, -1, -1, -1},
    {0, 11, 3, 0, 6, 11, 0, 9, 6, 5, 6, 9, 1, 2, 10, -1},
    {11, 8, 5, 11, 5, 6, 8, 0, 5, 10, 5, 2, 0, 2, 5, -1},
    {6, 11, 3, 6, 3, 5, 2, 10, 3, 10, 5, 3, -1, -1, -1, -1},
    {5, 8, 9, 5, 2, 8, 5, 6, 2, 3, 8, 2, -1, -1, -1, -1},
    {9, 5, 6, 9, 6, 0, 0, 6, 2, -1, -1, -1, -1, -1, -1, -1},
    {1, 5, 8, 1, 8, 0, 5, 6, 8, 3, 8, 2, 6, 2, 8, -1},
    {1, 5, 6, 2, 1, 6, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {1, 3, 6, 1, 6, 10, 3, 8, 6, 5, 6, 9, 8, 9, 6, -1},
    {10, 1, 0, 10, 0, 6, 9, 5, 0, 5, 6, 0, -1, -1, -1, -1},
    {0, 3, 8, 5, 6, 10, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {10, 5, 6, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {11, 5, 10, 7, 5, 11, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {11, 5, 10, 11, 7, 5, 8, 3, 0, -1, -1, -1, -1, -1, -1, -1},
    {5, 11, 7, 5, 10, 11, 1, 9, 0, -1, -1, -1, -1, -1, -1, -1},
    {10, 7, 5, 10, 11, 7, 9, 8, 1, 8, 3, 1, -1, -1, -1, -1},
    {11, 1, 2, 11, 7, 1, 7, 5, 1, -1, -1, -1, -1, -1, -1, -1},
    {0, 8, 3, 1, 2, 7, 1, 7, 5, 7, 2, 11, -1, -1, -1, -1},
    {9, 7, 5, 9, 2, 7, 9, 0, 2, 2, 11, 7, -1, -1, -1, -1},
    {7, 5, 2, 7, 2, 11, 5, 9, 2, 3, 2, 8, 9, 8, 2, -1},
    {2, 5, 10, 2, 3, 5, 3, 7, 5, -1, -1, -1, -1, -1, -1, -1},
    {8, 2, 0, 8, 5, 2, 8, 7, 5, 10, 2, 5, -1, -1, -1, -1},
    {9, 0, 1, 5, 10, 3, 5, 3, 7, 3, 10, 2, -1, -1, -1, -1},
    {9, 8, 2, 9, 2, 1, 8, 7, 2, 10, 2, 5, 7, 5, 2, -1},
    {1, 3, 5, 3, 7, 5, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 8, 7, 0, 7, 1, 1, 7, 5, -1, -1, -1, -1, -1, -1, -1},
    {9, 0, 3, 9, 3, 5, 5, 3, 7, -1, -1, -1, -1, -1, -1, -1},
    {9, 8, 7, 5, 9, 7, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {5, 8, 4, 5, 10, 8, 10, 11, 8, -1, -1, -1, -1, -1, -1, -1},
    {5, 0, 4, 5, 11, 0, 5, 10, 11, 11, 3, 0, -1, -1, -1, -1},
    {0, 1, 9, 8, 4, 10, 8, 10, 11, 10, 4, 5, -1, -1, -1, -1},
    {10, 11, 4, 10, 4, 5, 11, 3, 4, 9, 4, 1, 3, 1, 4, -1},
    {2, 5, 1, 2, 8, 5, 2, 11, 8, 4, 5, 8, -1, -1, -1, -1},
    {0, 4, 11, 0, 11, 3, 4, 5, 11, 2, 11, 1, 5, 1, 11, -1},
    {0, 2, 5, 0, 5, 9, 2, 11, 5, 4, 5, 8, 11, 8, 5, -1},
    {9, 4, 5, 2, 11, 3, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {2, 5, 10, 3, 5, 2, 3, 4, 5, 3, 8, 4, -1, -1, -1, -1},
    {5, 10, 2, 5, 2, 4, 4, 2, 0, -1, -1, -1, -1, -1, -1, -1},
    {3, 10, 2, 3, 5, 10, 3, 8, 5, 4, 5, 8, 0, 1, 9, -1},
    {5, 10, 2, 5, 2, 4, 1, 9, 2, 9, 4, 2, -1, -1, -1, -1},
    {8, 4, 5, 8, 5, 3, 3, 5, 1, -1, -1, -1, -1, -1, -1, -1},
    {0, 4, 5, 1, 0, 5, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {8, 4, 5, 8, 5, 3, 9, 0, 5, 0, 3, 5, -1, -1, -1, -1},
    {9, 4, 5, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {4, 11, 7, 4, 9, 11, 9, 10, 11, -1, -1, -1, -1, -1, -1, -1},
    {0, 8, 3, 4, 9, 7, 9, 11, 7, 9, 10, 11, -1, -1, -1, -1},
    {1, 10, 11, 1, 11, 4, 1, 4, 0, 7, 4, 11, -1, -1, -1, -1},
    {3, 1, 4, 3, 4, 8, 1, 10, 4, 7, 4, 11, 10, 11, 4, -1},
    {4, 11, 7, 9, 11, 4, 9, 2, 11, 9, 1, 2, -1, -1, -1, -1},
    {9, 7, 4, 9, 11, 7, 9, 1, 11, 2, 11, 1, 0, 8, 3, -1},
    {11, 7, 4, 11, 4, 2, 2, 4, 0, -1, -1, -1, -1, -1, -1, -1},
    {11, 7, 4, 11, 4, 2, 8, 3, 4, 3, 2, 4, -1, -1, -1, -1},
    {2, 9, 10, 2, 7, 9, 2, 3, 7, 7, 4, 9, -1, -1, -1, -1},
    {9, 10, 7, 9, 7, 4, 10, 2, 7, 8, 7, 0, 2, 0, 7, -1},
    {3, 7, 10, 3, 10, 2, 7, 4, 10, 1, 10, 0, 4, 0, 10, -1},
    {1, 10, 2, 8, 7, 4, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {4, 9, 1, 4, 1, 7, 7, 1, 3, -1, -1, -1, -1, -1, -1, -1},
    {4, 9, 1, 4, 1, 7, 0, 8, 1, 8, 7, 1, -1, -1, -1, -1},
    {4, 0, 3, 7, 4, 3, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {4, 8, 7, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {9, 10, 8, 10, 11, 8, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {3, 0, 9, 3, 9, 11, 11, 9, 10, -1, -1, -1, -1, -1, -1, -1},
    {0, 1, 10, 0, 10, 8, 8, 10, 11, -1, -1, -1, -1, -1, -1, -1},
    {3, 1, 10, 11, 3, 10, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {1, 2, 11, 1, 11, 9, 9, 11, 8, -1, -1, -1, -1, -1, -1, -1},
    {3, 0, 9, 3, 9, 11, 1, 2, 9, 2, 11, 9, -1, -1, -1, -1},
    {0, 2, 11, 8, 0, 11, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {3, 2, 11, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {2, 3, 8, 2, 8, 10, 10, 8, 9, -1, -1, -1, -1, -1, -1, -1},
    {9, 10, 2, 0, 9, 2, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {2, 3, 8, 2, 8, 10, 0, 1, 8, 1, 10, 8, -1, -1, -1, -1},
    {1, 10, 2, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {1, 3, 8, 9, 1, 8, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 9, 1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {0, 3, 8, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
    {-1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1},
};
__constant__ uint8_t kMcNtri[256] = {0, 1, 1, 2, 1, 2, 2, 3, 1, 2, 2, 3, 2, 3, 3, 2, 1, 2, 2, 3, 2, 3, 3, 4, 2, 3, 3, 4, 3, 4, 4, 3, 1, 2, 2, 3, 2, 3, 3, 4, 2, 3, 3, 4, 3, 4, 4, 3, 2, 3, 3, 2, 3, 4, 4, 3, 3, 4, 4, 3, 4, 5, 5, 2, 1, 2, 2, 3, 2, 3, 3, 4, 2, 3, 3, 4, 3, 4, 4, 3, 2, 3, 3, 4, 3, 4, 4, 5, 3, 4, 4, 5, 4, 5, 5, 4, 2, 3, 3, 4, 3, 4, 2, 3, 3, 4, 4, 5, 4, 5, 3, 2, 3, 4, 4, 3, 4, 5, 3, 2, 4, 5, 5, 4, 5, 2, 4, 1, 1, 2, 2, 3, 2, 3, 3, 4, 2, 3, 3, 4, 3, 4, 4, 3, 2, 3, 3, 4, 3, 4, 4, 5, 3, 2, 4, 3, 4, 3, 5, 2, 2, 3, 3, 4, 3, 4, 4, 5, 3, 4, 4, 5, 4, 5, 5, 4, 3, 4, 4, 3, 4, 5, 5, 4, 4, 3, 5, 2, 5, 4, 2, 1, 2, 3, 3, 4, 3, 4, 4, 5, 3, 4, 4, 5, 2, 3, 3, 2, 3, 4, 4, 5, 4, 5, 5, 2, 4, 3, 5, 4, 3, 2, 4, 1, 3, 4, 4, 5, 4, 5, 3, 4, 4, 5, 5, 2, 3, 4, 2, 1, 2, 3, 3, 2, 3, 4, 2, 1, 3, 2, 4, 1, 2, 1, 1, 0};

// Edges of a brick: edge (voxel v = x + 8y + 64z, axis a) is bit v + 512 a of
// kMcEdgeWords words.  A vertex belongs to the brick of its edge's low voxel,
// and its index is the brick's first plus its rank among the brick's edges.
constexpr int kMcEdgeBits = 3 * kVPB;
constexpr int kMcEdgeWords = kMcEdgeBits / 32;

// The 12 edges, 5 bits each: the low corner's offset (x + 2y + 4z), then the
// axis.  Looked up in a register: a chain of loads from the tables above per
// triangle corner would cost more than the corner.
constexpr unsigned long long mc_edge_pack()
{
    // kMcCorner[kMcEdgeLo[e]] and kMcEdgeAxis[e]
    constexpr int corner[8] = {0, 1, 3, 2, 4, 5, 7, 6};
    constexpr int lo[12] = {0, 1, 3, 0, 4, 5, 7, 4, 0, 1, 2, 3}, axis[12] = {0, 1, 0, 1, 0, 1, 0, 1, 2, 2, 2, 2};
    unsigned long long m = 0;
    for (int e = 0; e < 12; ++e)
        m |= (unsigned long long)(corner[lo[e]] | (axis[e] << 3)) << (5 * e);
    return m;
}
constexpr unsigned long long kMcEdges = mc_edge_pack();
__device__ __forceinline__ int mc_edge(int e) { return (int)(kMcEdges >> (5 * e)) & 31; }

// A brick's share of the mesh: triangles and vertices, and the sums of both
// over the bricks before it in its run of kMcRun bricks.
constexpr int kMcRun = 1024;
struct McBrick {
    uint32_t nt, nv, t0, v0;
};

// Key of the vertex on lattice edge (global voxel g, axis a): g biased by
// 2^18 per axis in bits 43-61 / 24-42 / 5-23, the axis in bits 0-4.
__device__ __forceinline__ unsigned long long mc_key(int gx, int gy, int gz, int a)
{
    return ((unsigned long long)(gx + kKeyBias) << 43) | ((unsigned long long)(gy + kKeyBias) << 24) |
           ((unsigned long long)(gz + kKeyBias) << 5) | (unsigned long long)a;
}

// Loads the voxels kLo .. 8 of brick b along each axis, from the brick and its
// neighbours, into tile (s, w), x fastest; a voxel of a missing or
// never-written brick reads (0, 0).  nb: the bricks at block offsets kLo / 8
// .. 1 (-1 where missing), x fastest.  A lookup compares 32-bit keys, and a
// missing block's key may be that of a brick elsewhere (alias_vector): the
// brick found is the neighbour only if its block is the one asked for.
// Starts and ends with a barrier.
template <typename T, int kLo, int kN>
__device__ void mc_load_tile(const GridView& g, unsigned int b, float2* tile, int* nb, int4& bc)
{
    constexpr int side = 9 - kLo, first = kLo < 0 ? -1 : 0, bs = 2 - first;
    __syncthreads();
    if (threadIdx.x < bs * bs * bs) {
        const int c = threadIdx.x;
        const int dx = c % bs + first, dy = c / bs % bs + first, dz = c / (bs * bs) + first;
        const int4 at = g.coords[b];
        int id = (dx | dy | dz) == 0 ? (int)b : find_brick(g, at.x + dx, at.y + dy, at.z + dz);
        if (id >= 0) {
            const int4 q = g.coords[id];
            if ((q.w & 1) || q.x != at.x + dx || q.y != at.y + dy || q.z != at.z + dz)
                id = -1;
        }
        nb[c] = id;
        if (c == 0)
            bc = at;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < side * side * side; i += kN) {
        const int x = i % side + kLo, y = i / side % side + kLo, z = i / (side * side) + kLo;
        const int id = nb[((x >> 3) - first) + bs * (((y >> 3) - first) + bs * ((z >> 3) - first))];
        float s = 0.f, w = 0.f;
        if (id >= 0)
            ld_pair((const T*)g.payload + (size_t)id * (2 * kVPB), (x & 7) + 8 * (y & 7) + 64 * (z & 7), s, w);
        tile[i] = make_float2(s, w);
    }
    __syncthreads();
}

// Case of the cell whose corner 0 is tile entry q; 0 when a corner is
// unobserved.
template <int kSide>
__device__ __forceinline__ int mc_case(const float2* tile, int q)
{
    int ci = 0;
    bool obs = true;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const int o = kMcCorner[k];
        const float2 v = tile[q + (o & 1) + kSide * (((o >> 1) & 1) + kSide * (o >> 2))];
        obs = obs && v.y != 0.0f;
        ci |= (v.x < 0.0f ? 1 : 0) << k;
    }
    return obs ? ci : 0;
}

__device__ __forceinline__ int mc_edge_mask(int ci)
{
    int m = 0;
#pragma unroll
    for (int e = 0; e < 12; ++e)
        m |= (((ci >> kMcEdgeLo[e]) ^ (ci >> kMcEdgeHi[e])) & 1) << e;
    return m;
}

// Inclusive sum over a workgroup of kN threads; *total gets the sum.
template <int kN, typename V>
__device__ __forceinline__ V mc_block_scan(V v, V* lds, V* total)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int o = 1; o < 64; o <<= 1) {
        const V u = __shfl_up(v, o);
        if (lane >= o)
            v += u;
    }
    if (lane == 63)
        lds[wv] = v;
    __syncthreads();
    V before = 0, all = 0;
    for (int k = 0; k < kN / 64; ++k) {
        before += k < wv ? lds[k] : (V)0;
        all += lds[k];
    }
    __syncthreads();
    *total = all;
    return v + before;
}

// Pass 1: every brick's triangles (kVPB / kMcCountThreads cells per thread, four), and the edges its
// cells use, set in the masks of the bricks that own them (cleared before).
// `uses` counts the edge uses.  Bound by the chain coords -> lookups -> tile
// of each brick: two wavefronts a brick keep more bricks in flight (room map,
// 33.5 k bricks: 84 us; 100 with four wavefronts, 93 with one, 170 with eight).
#ifndef TSDF_MC_COUNT_THREADS
#define TSDF_MC_COUNT_THREADS 128
#endif
constexpr int kMcCountThreads = TSDF_MC_COUNT_THREADS;

template <typename T>
__global__ __launch_bounds__(kMcCountThreads) void k_mc_count(GridView g, unsigned int n, McBrick* info, uint32_t* masks,
                                                       unsigned long long* uses)
{
    __shared__ float2 tile[9 * 9 * 9];
    __shared__ int nb[8];
    __shared__ int4 bc;
    __shared__ unsigned int red[kMcCountThreads / 64];
    __shared__ uint32_t used[8][kMcEdgeWords];
    unsigned int all_uses = 0;
    for (unsigned int b = blockIdx.x; b < n; b += gridDim.x) {
        for (int i = threadIdx.x; i < 8 * kMcEdgeWords; i += kMcCountThreads)
            (&used[0][0])[i] = 0u;
        mc_load_tile<T, 0, kMcCountThreads>(g, b, tile, nb, bc);
        unsigned int nt = 0;
        for (int k = 0; k < kVPB / kMcCountThreads; ++k) {
            const int cell = threadIdx.x + kMcCountThreads * k;
            const int x = cell & 7, y = (cell >> 3) & 7, z = cell >> 6;
            const int ci = mc_case<9>(tile, x + 9 * (y + 9 * z));
            if (ci == 0 || ci == 255)
                continue;
            nt += kMcNtri[ci];
            const int em = mc_edge_mask(ci);
            all_uses += (unsigned int)__popc(em);
#pragma unroll
            for (int e = 0; e < 12; ++e) {
                if (!((em >> e) & 1))
                    continue;
                const int o = kMcCorner[kMcEdgeLo[e]];
                const int ex = x + (o & 1), ey = y + ((o >> 1) & 1), ez = z + (o >> 2);
                const int v = (ex & 7) + 8 * (ey & 7) + 64 * (ez & 7) + kVPB * kMcEdgeAxis[e];
                atomicOr(&used[(ex >> 3) | ((ey >> 3) << 1) | ((ez >> 3) << 2)][v >> 5], 1u << (v & 31));
            }
        }
        unsigned int tt;
        mc_block_scan<kMcCountThreads>(nt, red, &tt);
        if (threadIdx.x == 0)
            info[b].nt = tt;
        if (tt)  // the scan's barriers ordered the LDS bits
            for (int i = threadIdx.x; i < 8 * kMcEdgeWords; i += kMcCountThreads) {
                const uint32_t m = (&used[0][0])[i];
                if (m)
                    atomicOr(&masks[(size_t)nb[i / kMcEdgeWords] * kMcEdgeWords + i % kMcEdgeWords], m);
            }
        __syncthreads();
    }
    all_uses = wave_sum(all_uses);
    if ((threadIdx.x & 63) == 0 && all_uses)
        atomicAdd(uses + (workgroup_index() % kStatLanes) * kStatStride, (unsigned long long)all_uses);
}

// Pass 2: vertices of every brick, sums within runs of kMcRun bricks, and the
// runs' totals.
__global__ __launch_bounds__(kMcRun) void k_mc_runs(unsigned int n, const uint32_t* masks, McBrick* info,
                                                    ulonglong2* runs)
{
    __shared__ unsigned int red[kMcRun / 64];
    const unsigned int b = blockIdx.x * kMcRun + threadIdx.x;
    unsigned int nt = 0, nv = 0;
    if (b < n) {
        nt = info[b].nt;
        const uint4* m = (const uint4*)(masks + (size_t)b * kMcEdgeWords);
        for (int k = 0; k < kMcEdgeWords / 4; ++k) {
            const uint4 q = m[k];
            nv += (unsigned int)(__popc(q.x) + __popc(q.y) + __popc(q.z) + __popc(q.w));
        }
    }
    unsigned int tt, tv;
    const unsigned int t1 = mc_block_scan<kMcRun>(nt, red, &tt), v1 = mc_block_scan<kMcRun>(nv, red, &tv);
    if (b < n)
        info[b] = McBrick{nt, nv, t1 - nt, v1 - nv};
    if (threadIdx.x == 0)
        runs[blockIdx.x] = make_ulonglong2(tt, tv);
}

// Pass 3: the runs' totals into the sums before each; totals[0..2]: triangles,
// vertices, edge uses.  One workgroup.
__global__ __launch_bounds__(kMcRun) void k_mc_totals(unsigned int n_runs, ulonglong2* runs,
                                                      const unsigned long long* uses, unsigned long long* totals)
{
    __shared__ unsigned long long red[kMcRun / 64];
    unsigned long long t0 = 0, v0 = 0;
    for (unsigned int r0 = 0; r0 < n_runs; r0 += kMcRun) {
        const unsigned int r = r0 + threadIdx.x;
        const ulonglong2 q = r < n_runs ? runs[r] : make_ulonglong2(0ull, 0ull);
        unsigned long long tt, tv;
        const unsigned long long t1 = mc_block_scan<kMcRun>((unsigned long long)q.x, red, &tt);
        const unsigned long long v1 = mc_block_scan<kMcRun>((unsigned long long)q.y, red, &tv);
        if (r < n_runs)
            runs[r] = make_ulonglong2(t0 + t1 - q.x, v0 + v1 - q.y);
        t0 += tt;
        v0 += tv;
    }
    if (threadIdx.x == 0) {
        unsigned long long u = 0;
        for (int k = 0; k < kStatLanes; ++k)
            u += uses[(size_t)k * kStatStride];
        totals[0] = t0;
        totals[1] = v0;
        totals[2] = u;
    }
}

// Pass 4: the mesh, brick by brick.  A brick writes the triangles of its cells
// and the vertices it owns.  Their normals need every cell around their edges,
// so the cells of the planes before the brick are taken again (729 for 512):
// the sums stay in LDS and nothing is accumulated in memory.
//
// Cases, owned edges and triangles are compacted into lists first: a few tens of
// a brick's 512 cells hold surface, and the fp64 work of the others' lanes
// would be idle.  262 us for the 2.28 M triangles and 1.15 M vertices of the
// room map (636 without the lists and with the tables in memory); as a global
// weld table (a hash insert per edge use, a lookup per triangle corner, 20 M
// fp64 atomics for the normals) the same work took 1.9 ms.
#ifndef TSDF_MC_EMIT_ROUNDS
#define TSDF_MC_EMIT_ROUNDS 8
#endif
constexpr int kMcSide = 10;  // voxels -1 .. 8

// Position of the vertex on edge (tile entry q, axis a) of global voxel gv,
// and the distances of its two ends.
__device__ __forceinline__ void mc_position(const float2* tile, int q, int a, const int (&gv)[3], double vl, double half,
                                            double (&p)[3], double& f0, double& f1)
{
    f0 = fabs((double)tile[q].x);
    f1 = fabs((double)tile[q + (a == 0 ? 1 : a == 1 ? kMcSide : kMcSide * kMcSide)].x);
    const double t = f0 * vl / (f0 + f1);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        p[k] = half + vl * (double)gv[k];
        p[k] = k == a ? p[k] + t : p[k];
    }
}

// Normals are summed in LDS for bricks of at most this many vertices (a noisy
// brick can have up to 1 536; 512 keep four workgroups on a CU), else in place
// in the output, which only this workgroup touches.
#ifndef TSDF_MC_ACC
#define TSDF_MC_ACC 512
#endif
constexpr int kMcAcc = TSDF_MC_ACC;

template <typename T, bool kColor>
__global__ __launch_bounds__(kThreads) void k_mc_emit(GridView g, unsigned int n, const McBrick* info,
                                                      const ulonglong2* runs, const uint32_t* masks, double* verts,
                                                      double* cols, double* vn, int32_t* faces,
                                                      unsigned long long* vkeys)
{
    constexpr int kCells = 9 * 9 * 9;  // cells -1 .. 7
    __shared__ float2 tile[kMcSide * kMcSide * kMcSide];
    __shared__ int nb[27];
    __shared__ int4 bc;
    __shared__ unsigned int red[kThreads / 64];
    __shared__ uint32_t used[8][kMcEdgeWords];  // edges of the brick and its + neighbours
    __shared__ uint16_t before[8][kMcEdgeWords];
    __shared__ uint32_t vfirst[8];
    __shared__ double acc[kMcAcc][3];  // face normals summed per owned vertex
    __shared__ int8_t tri[256][16];    // the case tables
    __shared__ uint8_t ntri[256];
    __shared__ uint8_t cases[kCells];
    __shared__ uint16_t first[kVPB];        // of the brick's cells: triangles before it
    __shared__ uint16_t list[5 * kCells];   // owned edges, then triangles (cell | number << 10)
    __shared__ unsigned int n_list;
    const double vl = (double)g.vl, half = vl * 0.5;
    for (int i = threadIdx.x; i < 256 * 16; i += kThreads)
        tri[i >> 4][i & 15] = kMcTri[i >> 4][i & 15];
    for (int i = threadIdx.x; i < 256; i += kThreads)
        ntri[i] = kMcNtri[i];
    for (unsigned int b = blockIdx.x; b < n; b += gridDim.x) {
        const McBrick me = info[b];
        if (me.nt == 0 && me.nv == 0)
            continue;
        const bool in_lds = me.nv <= (unsigned int)kMcAcc;
        mc_load_tile<T, -1, kThreads>(g, b, tile, nb, bc);
        for (int i = threadIdx.x; i < 8 * kMcEdgeWords; i += kThreads) {
            const int c = i / kMcEdgeWords;
            const int id = nb[((c & 1) + 1) + 3 * ((((c >> 1) & 1) + 1) + 3 * ((c >> 2) + 1))];
            (&used[0][0])[i] = id >= 0 ? masks[(size_t)id * kMcEdgeWords + i % kMcEdgeWords] : 0u;
            if (i % kMcEdgeWords == 0)
                vfirst[c] = id >= 0 ? (uint32_t)runs[id / kMcRun].y + info[id].v0 : 0u;
        }
        for (int i = threadIdx.x; i < kCells; i += kThreads)
            cases[i] = (uint8_t)mc_case<kMcSide>(tile, i % 9 + kMcSide * (i / 9 % 9 + kMcSide * (i / 81)));
        if (threadIdx.x == 0)
            n_list = 0;
        __syncthreads();
        // ranks: each wavefront scans the words of two bricks
        for (int c = threadIdx.x >> 6; c < 8; c += kThreads / 64) {
            const int lane = threadIdx.x & 63;
            const unsigned int own = lane < kMcEdgeWords ? (unsigned int)__popc(used[c][lane]) : 0u;
            unsigned int sum = own;
            for (int o = 1; o < 64; o <<= 1) {
                const unsigned int u = __shfl_up(sum, o);
                if (lane >= o)
                    sum += u;
            }
            if (lane < kMcEdgeWords) {
                before[c][lane] = (uint16_t)(sum - own);
                if (c == 0) {
                    unsigned int k = sum - own;
                    for (uint32_t m = used[0][lane]; m; m &= m - 1u)
                        list[k++] = (uint16_t)(32 * lane + __ffs(m) - 1);
                }
            }
        }
        // where the triangles of the brick's cells go (cell order)
        unsigned int own_t[2], nt = 0;
        for (int k = 0; k < 2; ++k) {
            const int cell = 2 * threadIdx.x + k;
            own_t[k] = ntri[cases[(cell & 7) + 1 + 9 * (((cell >> 3) & 7) + 1 + 9 * ((cell >> 6) + 1))]];
            nt += own_t[k];
        }
        unsigned int tot;
        const unsigned int t1 = mc_block_scan<kThreads>(nt, red, &tot) - nt;
        first[2 * threadIdx.x] = (uint16_t)t1;
        first[2 * threadIdx.x + 1] = (uint16_t)(t1 + own_t[0]);
        // the owned vertices
        for (unsigned int j = threadIdx.x; j < me.nv; j += kThreads) {
            const int e = list[j], a = e / kVPB, v = e & (kVPB - 1);
            const size_t id = (size_t)vfirst[0] + j;
            const int x = v & 7, y = (v >> 3) & 7, z = v >> 6;
            const int gv[3] = {bc.x * 8 + x, bc.y * 8 + y, bc.z * 8 + z};
            double p[3], f0, f1;
            mc_position(tile, (x + 1) + kMcSide * ((y + 1) + kMcSide * (z + 1)), a, gv, vl, half, p, f0, f1);
            for (int k = 0; k < 3; ++k)
                verts[3 * id + k] = p[k];
            if (kColor) {
                const int hx = x + (a == 0), hy = y + (a == 1), hz = z + (a == 2);
                const int hi = nb[((hx >> 3) + 1) + 3 * (((hy >> 3) + 1) + 3 * ((hz >> 3) + 1))];
                const int hv = (hx & 7) + 8 * (hy & 7) + 64 * (hz & 7);
                for (int k = 0; k < 3; ++k) {
                    const double c0 = (double)g.rgb[((size_t)b * 3 + k) * kVPB + v] / 255.0;
                    const double c1 = (double)g.rgb[((size_t)hi * 3 + k) * kVPB + hv] / 255.0;
                    cols[3 * id + k] = (f1 * c0 + f0 * c1) / (f0 + f1);
                }
            }
            if (vkeys)
                vkeys[id] = mc_key(gv[0], gv[1], gv[2], a);
            if (vn)
                for (int k = 0; k < 3; ++k)
                    (in_lds ? acc[j] : vn + 3 * id)[k] = 0.0;
        }
        __syncthreads();
        // the triangles to take: the brick's own, and with normals those of
        // the cells before it
        const bool halo = vn && me.nv;
        for (int i = threadIdx.x; i < kCells; i += kThreads) {
            const int m = ntri[cases[i]];
            if (m == 0 || (!halo && (i % 9 == 0 || i / 9 % 9 == 0 || i < 81)))
                continue;
            const unsigned int at = atomicAdd(&n_list, (unsigned int)m);
            for (int q = 0; q < m; ++q)
                list[at + q] = (uint16_t)(i | (q << 10));
        }
        __syncthreads();
        const size_t tfirst = (size_t)runs[b / kMcRun].x + me.t0;
        for (unsigned int j = threadIdx.x; j < n_list; j += kThreads) {
            const int i = list[j] & 1023, q = list[j] >> 10, cs = cases[i];
            const int x = i % 9 - 1, y = i / 9 % 9 - 1, z = i / 81 - 1;
            const int q0 = (x + 1) + kMcSide * ((y + 1) + kMcSide * (z + 1));
            const bool mine = (x | y | z) >= 0;
            double p[3][3];
            int slot[3];
#pragma unroll
            for (int r = 0; r < 3; ++r) {
                // table order e0, e2, e1
                const int e = mc_edge(tri[cs][3 * q + (r == 0 ? 0 : 3 - r)]), o = e & 7, a = e >> 3;
                const int ex = x + (o & 1), ey = y + ((o >> 1) & 1), ez = z + (o >> 2);
                // the edge's brick among used[], when it is no brick before this one
                const int c = (ex >> 3 & 1) | ((ey >> 3 & 1) << 1) | ((ez >> 3 & 1) << 2);
                const int v = (ex & 7) + 8 * (ey & 7) + 64 * (ez & 7) + kVPB * a;
                const int rank = (int)before[c][v >> 5] + __popc(used[c][v >> 5] & ((1u << (v & 31)) - 1u));
                slot[r] = ((ex | ey | ez) & ~7) == 0 ? rank : -1;
                if (mine)
                    faces[3 * (tfirst + first[x + 8 * y + 64 * z] + q) + r] = (int32_t)(vfirst[c] + rank);
                if (halo) {
                    const int gv[3] = {bc.x * 8 + ex, bc.y * 8 + ey, bc.z * 8 + ez};
                    double f0, f1;
                    mc_position(tile, q0 + (o & 1) + kMcSide * (((o >> 1) & 1) + kMcSide * (o >> 2)), a, gv, vl, half,
                                p[r], f0, f1);
                }
            }
            if (halo) {
                double u[3], w[3];
                for (int k = 0; k < 3; ++k) {
                    u[k] = p[1][k] - p[0][k];
                    w[k] = p[2][k] - p[0][k];
                }
                const double nrm[3] = {u[1] * w[2] - u[2] * w[1], u[2] * w[0] - u[0] * w[2], u[0] * w[1] - u[1] * w[0]};
#pragma unroll
                for (int r = 0; r < 3; ++r)
                    if (slot[r] >= 0)
                        for (int k = 0; k < 3; ++k) {
                            if (in_lds)
                                unsafeAtomicAdd(&acc[slot[r]][k], nrm[k]);
                            else
                                unsafeAtomicAdd(&vn[3 * ((size_t)vfirst[0] + slot[r]) + k], nrm[k]);
                        }
            }
        }
        if (!halo)
            continue;
        __syncthreads();
        // unit normals (Eigen's normalize: a zero vector stays zero)
        for (unsigned int j = threadIdx.x; j < me.nv; j += kThreads) {
            double* o = vn + 3 * ((size_t)vfirst[0] + j);
            double p[3];
            for (int k = 0; k < 3; ++k)
                p[k] = in_lds ? acc[j][k] : __hip_atomic_load(o + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const double z = p[0] * p[0] + p[1] * p[1] + p[2] * p[2];
            if (z > 0.0) {
                const double r = sqrt(z);
                p[0] /= r;
                p[1] /= r;
                p[2] /= r;
            }
            for (int k = 0; k < 3; ++k)
                o[k] = p[k];
        }
    }
}

__global__ __launch_bounds__(kThreads) void k_fill_u128(uint4* p, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = make_uint4(0u, 0u, 0u, 0u);
}

}  // namespace

extern "C" {

tsdf_status tsdf_marching_cubes(tsdf_grid* g, double* vertices, double* vertex_colors, double* vertex_normals,
                                int32_t* triangles, uint64_t* vertex_keys, uint64_t vertex_cap, uint64_t triangle_cap,
                                uint64_t* n_vertices, uint64_t* n_triangles, void* stream)
{
    if (!g || !n_vertices || !n_triangles)
        return fail(TSDF_BAD_ARG, "NULL grid or count");
    if ((vertex_cap && !vertices) || (triangle_cap && !triangles))
        return fail(TSDF_BAD_ARG, "NULL vertex or triangle buffer with a nonzero capacity");
    if (vertex_colors && !g->rgb)
        return fail(TSDF_BAD_ARG, "vertex colours asked of a grid without colour");
    DeviceScope ds(g->p.device);
    hipStream_t s = (hipStream_t)stream;
    HIPC(hipMemcpyAsync(g->ctrl_host, g->ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, s));
    HIPC(hipStreamSynchronize(s));
    *n_vertices = 0;
    *n_triangles = 0;
    const Ctrl& c = *g->ctrl_host;
    const unsigned int n = c.alloc_top < g->p.n_bricks ? c.alloc_top : g->p.n_bricks;
    if (n == 0)
        return TSDF_OK;
    // every block ever inserted lies in the control block's bounding box
    for (int a = 0; a < 3; ++a)
        if (c.bbox_min[a] < -(kKeyBias / 8) || c.bbox_max[a] >= kKeyBias / 8 - 1)
            return fail(TSDF_BAD_ARG, "map extent beyond the vertex key range (+-32767 blocks per axis)");
    const bool f16 = g->p.storage == TSDF_STORAGE_F16;
    const int bgrid = (int)(n < 65536u ? n : 65536u);
    const int egrid = (int)std::min(n, (unsigned int)g->n_cu * 4u * TSDF_MC_EMIT_ROUNDS);  // 4 workgroups fit a CU
    const unsigned int n_runs = (n + kMcRun - 1) / kMcRun;
    // one buffer: edge masks and edge-use lanes (cleared), the bricks' shares,
    // the runs' sums, the totals
    const size_t mask_b = (size_t)n * kMcEdgeWords * sizeof(uint32_t), uses_b = (size_t)kStatLanes * kStatStride * 8;
    const size_t info_b = (size_t)n * sizeof(McBrick), runs_b = (size_t)n_runs * sizeof(ulonglong2);
    const size_t need = mask_b + uses_b + info_b + runs_b + 4 * sizeof(unsigned long long);
    if (g->mc_cap < need) {
        HIPC(hipStreamSynchronize(s));
        (void)hipFree(g->mc_buf);
        g->mc_buf = nullptr;
        g->mc_cap = 0;
        HIPC(hipMalloc(&g->mc_buf, need));
        g->mc_cap = need;
    }
    uint32_t* masks = (uint32_t*)g->mc_buf;
    unsigned long long* uses = (unsigned long long*)((char*)g->mc_buf + mask_b);
    McBrick* info = (McBrick*)((char*)uses + uses_b);
    ulonglong2* runs = (ulonglong2*)((char*)info + info_b);
    unsigned long long* totals = (unsigned long long*)((char*)runs + runs_b);
    hipLaunchKernelGGL(k_fill_u128, dim3(g->n_cu * 4), dim3(kThreads), 0, s, (uint4*)masks, (mask_b + uses_b) / 16);
    if (f16)
        hipLaunchKernelGGL(k_mc_count<__half>, dim3(bgrid), dim3(kMcCountThreads), 0, s, view(g), n, info, masks, uses);
    else
        hipLaunchKernelGGL(k_mc_count<float>, dim3(bgrid), dim3(kMcCountThreads), 0, s, view(g), n, info, masks, uses);
    hipLaunchKernelGGL(k_mc_runs, dim3(n_runs), dim3(kMcRun), 0, s, n, masks, info, runs);
    hipLaunchKernelGGL(k_mc_totals, dim3(1), dim3(kMcRun), 0, s, n_runs, runs, uses, totals);
    HIPC(hipGetLastError());
    unsigned long long* tot = g->stat_host;  // pinned
    HIPC(hipMemcpyAsync(tot, totals, 3 * sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    HIPC(hipStreamSynchronize(s));
    const unsigned long long T = tot[0], V = tot[1], E = tot[2];
    if (E > 1ull << 31)
        return fail(TSDF_BAD_ARG, "mesh too large for 32-bit vertex indices");
    if (T > 0 && V <= vertex_cap && T <= triangle_cap) {
        auto emit = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(egrid), dim3(kThreads), 0, s, view(g), n, info, runs, masks, vertices,
                               vertex_colors, vertex_normals, triangles, (unsigned long long*)vertex_keys);
        };
        if (vertex_colors)
            f16 ? emit(k_mc_emit<__half, true>) : emit(k_mc_emit<float, true>);
        else
            f16 ? emit(k_mc_emit<__half, false>) : emit(k_mc_emit<float, false>);
        HIPC(hipGetLastError());
        HIPC(hipStreamSynchronize(s));
    }
    *n_vertices = V;
    *n_triangles = T;
    return TSDF_OK;
}

}  // extern "C"
