// tsdf_maintain.hpp -- map maintenance and surface extraction: erase empty
// bricks (cleanMemory) and a triangle mesh of the zero level set.  Included
// once, at the end of tsdf_hip.hip.
//
// cleanMemory / cleanTag, GPUVoxelGrid.cpp:185-196, 785-805: every brick whose
// 512 weights are all zero leaves the map.  Here the n surviving bricks get
// the ids 0..n-1 (ids are not observable): those with greater ids move into
// the free ones below n, the others stay, and the table is rebuilt.  All of it
// is decided on the device; the host waits once, for the count.
//
// marchingCubesHost, GPUVoxelGrid.cpp:200-251, copies the bricks into an
// Open3D ScalableTSDFVolume and calls its ExtractTriangleMesh on the host.
// Here the mesh is extracted on the GPU by marching tetrahedra: every cell of
// 8 voxel centres (x..x+1, y..y+1, z..z+1), all observed (w > 0), is split
// into 6 tetrahedra around its diagonal from corner 0 to corner 7 (corner
// c = (c & 1, c >> 1 & 1, c >> 2 & 1)); the same split in every cell makes
// neighbouring cells agree on their shared faces, so the surface is closed
// wherever the field is observed.  Vertices lie on tetrahedron edges whose
// ends change sign, at p = pa + t (pb - pa), t = sa / (sa - sb) with a the
// inside (sdf < 0) corner, so neighbours compute shared vertices bit for bit;
// each triangle faces the positive (free-space) side.
#pragma once

namespace {

// ---------------------------------------------------------------------------
// clean
// ---------------------------------------------------------------------------
struct CleanState {
    unsigned int dead;    // bricks that leave
    unsigned int n;       // bricks before
    unsigned int holes;   // dead ids below the surviving count ...
    unsigned int movers;  // ... and surviving ids at or above it: as many
};

__global__ void k_clean_begin(GridView g, CleanState* st)
{
    *st = CleanState{0u, min(g.ctrl->alloc_top, g.n_bricks), 0u, 0u};
}

// One wavefront per brick.  Bound by memory: most bricks show a weight in
// their first quarter, so the rest is read only where that one has none.
// 17 k fp32 bricks: 25.5 us when each was read whole by 8-byte loads, 11 now.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_alive(GridView g, CleanState* st, uint8_t* alive)
{
    constexpr int kPairs = sizeof(T) == 4 ? 2 : 4;           // (sdf, w) pairs in 16 bytes
    constexpr int kRounds = kVPB / (64 * kPairs);
    __shared__ unsigned int s_dead;
    if (threadIdx.x == 0)
        s_dead = 0u;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const unsigned int n = st->n, nw = gridDim.x * (kThreads / 64);
    auto observed = [](const uint4& q) {
        if constexpr (sizeof(T) == 4)
            return __uint_as_float(q.y) != 0.0f || __uint_as_float(q.w) != 0.0f;
        else  // the high halves; -0 is zero
            return ((q.x | q.y | q.z | q.w) & 0x7FFF0000u) != 0u;
    };
    for (unsigned int b = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6); b < n; b += nw) {
        const uint4* q = (const uint4*)((const T*)g.payload + (size_t)b * (2 * kVPB)) + lane;
        const bool fresh = (g.coords[b].w & 1) != 0;  // allocated, never written: all zero
        bool any = __ballot(observed(q[0])) != 0ull;
        if (!any) {
            bool more = false;
#pragma unroll
            for (int r = 1; r < kRounds; ++r)
                more |= observed(q[r * 64]);
            any = __ballot(more) != 0ull;
        }
        if (lane == 0) {
            alive[b] = any && !fresh ? 1 : 0;
            if (!any || fresh)
                atomicAdd(&s_dead, 1u);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0 && s_dead)
        atomicAdd(&st->dead, s_dead);
}

// Lists the moves and clears the table, its superblock bits and its box.
// Nothing to do where every brick stays.
__global__ __launch_bounds__(kThreads) void k_clean_plan(GridView g, CleanState* st, const uint8_t* alive,
                                                         uint32_t* hole, uint32_t* mover)
{
    if (st->dead == 0u)
        return;
    const unsigned int n = st->n, kept = n - st->dead;
    const unsigned int t0 = blockIdx.x * kThreads + threadIdx.x, step = gridDim.x * kThreads;
    for (unsigned int i = t0; i < n; i += step) {
        const bool a = alive[i] != 0;
        if (i < kept && !a)
            hole[atomicAdd(&st->holes, 1u)] = i;
        if (i >= kept && a)
            mover[atomicAdd(&st->movers, 1u)] = i;
    }
    for (size_t i = t0; i <= g.mask; i += step) {
        g.slots[i] = kSlotEmpty;
        g.slot_epoch[i] = 0u;
    }
    for (size_t i = t0; i < kSbWords; i += step)
        g.sb_bits[i] = 0u;
    if (t0 == 0) {
        for (int a = 0; a < 3; ++a) {
            g.ctrl->bbox_min[a] = 0x7FFFFFFF;
            g.ctrl->bbox_max[a] = (int)0x80000000u;
        }
        g.ctrl->sb_version += 1u;  // the bits are rebuilt
        g.ctrl->alloc_top = kept;
    }
}

// Enters brick `id` at block c into the table (as prime_hash's key) and the
// superblock bits.
__device__ __forceinline__ void rehash(const GridView& g, const int4& c, unsigned int id)
{
    const uint32_t key = prime_hash(c.x, c.y, c.z);
    const unsigned long long word = ((unsigned long long)key << 32) | id;
    uint32_t b = mix32(key) & g.mask;
    for (uint32_t p = 0; p <= g.mask; ++p) {
        if (atomicCAS(&g.slots[b], kSlotEmpty, word) == kSlotEmpty)
            break;
        b = (b + 1) & g.mask;
    }
    // 512 blocks share a bit and neighbours come together, so one lane sets it
    // for all that have the same (an atomic each, 17 k on a few words: 32 us
    // for the kernel, 19 now)
    const int sb = sb_index(c.x, c.y, c.z);
    for (bool todo = sb >= 0; todo;) {
        const int first = __builtin_amdgcn_readfirstlane(sb);
        if (sb == first) {
            if (__ffsll((unsigned long long)__ballot(1)) - 1 == (int)__lane_id())
                atomicOr(&g.sb_bits[sb >> 5], 1u << (sb & 31));
            todo = false;
        }
    }
}

// Moves the listed bricks (a wavefront each, 16 bytes a lane; sources and
// destinations are disjoint) and enters every survivor into the table.  The
// box is reduced over the workgroup first: six atomics each on one address.
__global__ __launch_bounds__(kThreads) void k_clean_apply(GridView g, const CleanState* st, const uint8_t* alive,
                                                          const uint32_t* hole, const uint32_t* mover, int payload16)
{
    if (st->dead == 0u)
        return;
    __shared__ int box[6];  // least x, y, z; greatest x, y, z, complemented
    if (threadIdx.x < 6)
        box[threadIdx.x] = 0x7FFFFFFF;
    __syncthreads();
    const unsigned int kept = st->n - st->dead, moves = st->holes;
    const int lane = threadIdx.x & 63;
    int3 mn = make_int3(0x7FFFFFFF, 0x7FFFFFFF, 0x7FFFFFFF);
    int3 mx = make_int3((int)0x80000000u, (int)0x80000000u, (int)0x80000000u);
    auto enter = [&](const int4& c, unsigned int id) {
        rehash(g, c, id);
        mn = make_int3(min(mn.x, c.x), min(mn.y, c.y), min(mn.z, c.z));
        mx = make_int3(max(mx.x, c.x), max(mx.y, c.y), max(mx.z, c.z));
    };
    for (unsigned int j = blockIdx.x * kThreads + threadIdx.x; j < kept; j += gridDim.x * kThreads)
        if (alive[j])
            enter(g.coords[j], j);
    const unsigned int nw = gridDim.x * (kThreads / 64);
    for (unsigned int m = blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6); m < moves; m += nw) {
        const unsigned int to = hole[m], from = mover[m];
        uint4* const p = (uint4*)g.payload;
        for (int k = lane; k < payload16; k += 64)
            p[(size_t)to * payload16 + k] = p[(size_t)from * payload16 + k];
        if (g.rgb) {
            constexpr int kRgb16 = 3 * kVPB / 4;
            uint4* const r = (uint4*)g.rgb;
            for (int k = lane; k < kRgb16; k += 64)
                r[(size_t)to * kRgb16 + k] = r[(size_t)from * kRgb16 + k];
        }
        if (lane == 0) {
            const int4 c = g.coords[from];
            g.coords[to] = c;
            enter(c, to);
        }
    }
    if (mn.x <= mx.x) {
        atomicMin(&box[0], mn.x);
        atomicMin(&box[1], mn.y);
        atomicMin(&box[2], mn.z);
        atomicMin(&box[3], ~mx.x);
        atomicMin(&box[4], ~mx.y);
        atomicMin(&box[5], ~mx.z);
    }
    __syncthreads();
    if (threadIdx.x < 3 && box[threadIdx.x] <= ~box[threadIdx.x + 3])
        atomicMin(&g.ctrl->bbox_min[threadIdx.x], box[threadIdx.x]);
    else if (threadIdx.x >= 3 && threadIdx.x < 6 && box[threadIdx.x - 3] <= ~box[threadIdx.x])
        atomicMax(&g.ctrl->bbox_max[threadIdx.x - 3], ~box[threadIdx.x]);
}

__global__ void k_fill_u64(unsigned long long* p, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = 0ull;
}

// ---------------------------------------------------------------------------
// mesh
// ---------------------------------------------------------------------------

// The 6 tetrahedra of a cell, corners by index c = x + 2y + 4z.
__constant__ int kTets[6][4] = {{0, 1, 3, 7}, {0, 3, 2, 7}, {0, 2, 6, 7}, {0, 6, 4, 7}, {0, 4, 5, 7}, {0, 5, 1, 7}};

// A triangle as the three tetrahedron edges its vertices lie on: vertex q is
// on the edge from inside corner a[q] to outside corner b[q].
struct TriEdges {
    int8_t a[3], b[3];
};

__device__ __forceinline__ void edge_point(const float (&p)[8][3], const float (&s)[8], int a, int b, float* out)
{
    const float t = s[a] / (s[a] - s[b]);
#pragma unroll
    for (int k = 0; k < 3; ++k)
        out[k] = p[a][k] + t * (p[b][k] - p[a][k]);
}

// Triangles of tetrahedron `tet` of a cell; returns how many (0..2).
__device__ __forceinline__ int tet_triangles(const float (&p)[8][3], const float (&s)[8], int tet, TriEdges* out)
{
    const int c[4] = {kTets[tet][0], kTets[tet][1], kTets[tet][2], kTets[tet][3]};
    int in[4], out_[4], ni = 0, no = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (s[c[k]] < 0.0f)
            in[ni++] = c[k];
        else
            out_[no++] = c[k];
    }
    if (ni == 0 || no == 0)
        return 0;
    int nt;
    if (ni == 1) {
        out[0] = TriEdges{{(int8_t)in[0], (int8_t)in[0], (int8_t)in[0]},
                          {(int8_t)out_[0], (int8_t)out_[1], (int8_t)out_[2]}};
        nt = 1;
    } else if (no == 1) {
        out[0] = TriEdges{{(int8_t)in[0], (int8_t)in[1], (int8_t)in[2]},
                          {(int8_t)out_[0], (int8_t)out_[0], (int8_t)out_[0]}};
        nt = 1;
    } else {
        // the quad e00 e01 e11 e10 (e_ij: inside i to outside j) as two triangles
        out[0] = TriEdges{{(int8_t)in[0], (int8_t)in[0], (int8_t)in[1]},
                          {(int8_t)out_[0], (int8_t)out_[1], (int8_t)out_[1]}};
        out[1] = TriEdges{{(int8_t)in[0], (int8_t)in[1], (int8_t)in[1]},
                          {(int8_t)out_[0], (int8_t)out_[1], (int8_t)out_[0]}};
        nt = 2;
    }
    // face the free-space side: from the inside corners toward the outside
    float d[3] = {0.f, 0.f, 0.f};
    for (int k = 0; k < ni; ++k)
        for (int q = 0; q < 3; ++q)
            d[q] -= p[in[k]][q] / (float)ni;
    for (int k = 0; k < no; ++k)
        for (int q = 0; q < 3; ++q)
            d[q] += p[out_[k]][q] / (float)no;
    for (int t = 0; t < nt; ++t) {
        float v0[3], v1[3], v2[3];
        edge_point(p, s, out[t].a[0], out[t].b[0], v0);
        edge_point(p, s, out[t].a[1], out[t].b[1], v1);
        edge_point(p, s, out[t].a[2], out[t].b[2], v2);
        const float a[3] = {v1[0] - v0[0], v1[1] - v0[1], v1[2] - v0[2]};
        const float b[3] = {v2[0] - v0[0], v2[1] - v0[1], v2[2] - v0[2]};
        const float n[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]};
        if (n[0] * d[0] + n[1] * d[1] + n[2] * d[2] < 0.0f) {
            const int8_t ta = out[t].a[1], tb = out[t].b[1];
            out[t].a[1] = out[t].a[2];
            out[t].b[1] = out[t].b[2];
            out[t].a[2] = ta;
            out[t].b[2] = tb;
        }
    }
    return nt;
}

// Key of the vertex on the edge from voxel (gx, gy, gz) (inside) to its
// neighbour at offset (dx, dy, dz) (outside): the voxel's global index,
// biased by 2^18 per axis (19 bits each), and the offset (5 bits).  Equal
// keys are equal vertices bit for bit.
constexpr int kKeyBias = 1 << 18;

__device__ __forceinline__ unsigned long long vertex_key(int gx, int gy, int gz, int dx, int dy, int dz)
{
    return ((unsigned long long)(gx + kKeyBias) << 43) | ((unsigned long long)(gy + kKeyBias) << 24) |
           ((unsigned long long)(gz + kKeyBias) << 5) | (unsigned long long)((dx + 1) + 3 * (dy + 1) + 9 * (dz + 1));
}

// One workgroup per brick, two cells per thread.  tris: [cap][3][3] world
// coordinates; cols (kColor): [cap][3][3] vertex colours interpolated like
// the positions; keys (or null): [cap][3] vertex keys; count: total
// triangles (may exceed cap).  A brick that was allocated but never written
// (coords.w bit 0) counts as unobserved.
template <typename T, bool kColor>
__global__ __launch_bounds__(kThreads) void k_mesh(GridView g, unsigned int n, float* tris, float* cols,
                                                   unsigned long long* keys, unsigned long long cap,
                                                   unsigned long long* count)
{
    __shared__ int nb[8];  // brick ids of (dx, dy, dz) = (c & 1, c >> 1 & 1, c >> 2 & 1)
    __shared__ int4 bc;
    for (unsigned int b = blockIdx.x; b < n; b += gridDim.x) {
        __syncthreads();
        if (threadIdx.x == 0)
            bc = g.coords[b];
        __syncthreads();
        if (threadIdx.x < 8) {
            const int c = threadIdx.x;
            int id = c == 0 ? (int)b : find_brick(g, bc.x + (c & 1), bc.y + ((c >> 1) & 1), bc.z + ((c >> 2) & 1));
            if (id >= 0 && (g.coords[id].w & 1))
                id = -1;
            nb[c] = id;
        }
        __syncthreads();
        for (int cell = threadIdx.x; cell < kVPB; cell += kThreads) {
            const int x = cell & 7, y = (cell >> 3) & 7, z = cell >> 6;
            float s[8], p[8][3];
            int vid[8], vbrick[8];
            bool ok = true;
#pragma unroll
            for (int c = 0; c < 8; ++c) {
                const int vx = x + (c & 1), vy = y + ((c >> 1) & 1), vz = z + ((c >> 2) & 1);
                const int which = (vx >> 3) | ((vy >> 3) << 1) | ((vz >> 3) << 2);
                const int id = nb[which];
                const int v = (vx & 7) + 8 * (vy & 7) + 64 * (vz & 7);
                float w = 0.f, sv = 0.f;
                if (id >= 0)
                    ld_pair((const T*)g.payload + (size_t)id * (2 * kVPB), v, sv, w);
                ok = ok && id >= 0 && w > 0.0f;
                s[c] = sv;
                vid[c] = v;
                vbrick[c] = id;
                p[c][0] = voxel_mid(vx & 7, bc.x + (vx >> 3), g.vbl, g.vl);
                p[c][1] = voxel_mid(vy & 7, bc.y + (vy >> 3), g.vbl, g.vl);
                p[c][2] = voxel_mid(vz & 7, bc.z + (vz >> 3), g.vbl, g.vl);
            }
            TriEdges tri[12];
            int nt = 0;
            if (ok)
                for (int t = 0; t < 6; ++t)
                    nt += tet_triangles(p, s, t, tri + nt);
            // wave-aggregated slots in the output
            int incl = nt;
            for (int o = 1; o < 64; o <<= 1) {
                const int v = __shfl_up(incl, o);
                if ((int)__lane_id() >= o)
                    incl += v;
            }
            const int total = __shfl(incl, 63);
            unsigned long long base = 0;
            if (__lane_id() == 63 && total)
                base = atomicAdd(count, (unsigned long long)total);
            base = __shfl(base, 63);
            const unsigned long long first = base + (unsigned long long)(incl - nt);
            for (int t = 0; t < nt; ++t) {
                const unsigned long long k = first + t;
                if (k >= cap)
                    break;
                for (int q = 0; q < 3; ++q) {
                    const int a = tri[t].a[q], bb = tri[t].b[q];
                    float v[3];
                    edge_point(p, s, a, bb, v);
                    for (int r = 0; r < 3; ++r)
                        tris[k * 9 + q * 3 + r] = v[r];
                    if (keys) {
                        const int ax = a & 1, ay = (a >> 1) & 1, az = (a >> 2) & 1;
                        keys[k * 3 + q] = vertex_key(bc.x * 8 + x + ax, bc.y * 8 + y + ay, bc.z * 8 + z + az,
                                                     (bb & 1) - ax, ((bb >> 1) & 1) - ay, ((bb >> 2) & 1) - az);
                    }
                    if (kColor) {
                        const float u = s[a] / (s[a] - s[bb]);
                        const float* ca = g.rgb + (size_t)vbrick[a] * 3 * kVPB + vid[a];
                        const float* cb = g.rgb + (size_t)vbrick[bb] * 3 * kVPB + vid[bb];
                        for (int r = 0; r < 3; ++r) {
                            const float x0 = ca[r * kVPB], x1 = cb[r * kVPB];
                            cols[k * 9 + q * 3 + r] = x0 + u * (x1 - x0);
                        }
                    }
                }
            }
        }
    }
}

}  // namespace

extern "C" {

tsdf_status tsdf_clean(tsdf_grid* g, uint64_t* n_removed, void* stream)
{
    if (!g)
        return fail(TSDF_BAD_ARG, "NULL grid");
    if (n_removed)
        *n_removed = 0;
    DeviceScope ds(g->p.device);
    hipStream_t s = (hipStream_t)stream;
    // the state, both move lists (a move takes a dead and a surviving brick,
    // so at most half of the pool each) and a flag per brick
    const size_t half = ((size_t)g->p.n_bricks + 1) / 2;
    if (!g->clean_buf)
        HIPC(hipMalloc(&g->clean_buf, sizeof(CleanState) + 2 * half * sizeof(uint32_t) + g->p.n_bricks));
    CleanState* st = (CleanState*)g->clean_buf;
    uint32_t* hole = (uint32_t*)(st + 1);
    uint32_t* mover = hole + half;
    uint8_t* alive = (uint8_t*)(mover + half);
    ++g->map_gen;  // the table and superblock bits are rebuilt
    const bool f16 = g->p.storage == TSDF_STORAGE_F16;
    const int payload16 = 2 * kVPB * (int)(f16 ? sizeof(__half) : sizeof(float)) / 16;
    const dim3 grid(g->n_cu * 8), threads(kThreads);
    hipLaunchKernelGGL(k_clean_begin, dim3(1), dim3(1), 0, s, view(g), st);
    if (f16)
        hipLaunchKernelGGL(k_alive<__half>, grid, threads, 0, s, view(g), st, alive);
    else
        hipLaunchKernelGGL(k_alive<float>, grid, threads, 0, s, view(g), st, alive);
    hipLaunchKernelGGL(k_clean_plan, grid, threads, 0, s, view(g), st, alive, hole, mover);
    hipLaunchKernelGGL(k_clean_apply, grid, threads, 0, s, view(g), st, alive, hole, mover, payload16);
    HIPC(hipGetLastError());
    HIPC(hipMemcpyAsync(g->stat_host, st, sizeof(CleanState), hipMemcpyDeviceToHost, s));
    HIPC(hipStreamSynchronize(s));
    if (n_removed)
        *n_removed = ((const CleanState*)g->stat_host)->dead;
    return TSDF_OK;
}

tsdf_status tsdf_extract_mesh(tsdf_grid* g, float* triangles, float* colors, uint64_t* vertex_keys, uint64_t cap,
                              uint64_t* n_triangles, void* stream)
{
    if (!g || !n_triangles || (cap && !triangles))
        return fail(TSDF_BAD_ARG, "NULL grid, count or triangle buffer");
    if (colors && !g->rgb)
        return fail(TSDF_BAD_ARG, "vertex colours asked of a grid without colour");
    tsdf_stats_out st;
    tsdf_status r = tsdf_stats(g, &st, stream);
    if (r != TSDF_OK)
        return r;
    *n_triangles = 0;
    const unsigned int n = (unsigned int)st.n_bricks;
    if (n == 0)
        return TSDF_OK;
    if (vertex_keys) {
        // every block ever inserted lies in the control block's bounding box
        const Ctrl& c = *g->ctrl_host;
        for (int a = 0; a < 3; ++a)
            if (c.bbox_min[a] < -(kKeyBias / 8) || c.bbox_max[a] >= kKeyBias / 8 - 1)
                return fail(TSDF_BAD_ARG, "map extent beyond the vertex key range (+-32767 blocks per axis)");
    }
    DeviceScope ds(g->p.device);
    hipStream_t s = (hipStream_t)stream;
    unsigned long long* cnt = nullptr;
    HIPC(hipMalloc(&cnt, sizeof(unsigned long long)));
    hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(1), 0, s, cnt, (size_t)1);
    unsigned long long* keys = cap > 0 ? (unsigned long long*)vertex_keys : nullptr;
    const int grid = (int)(n < 65536u ? n : 65536u);
    const bool f16 = g->p.storage == TSDF_STORAGE_F16;
    const bool col = colors != nullptr && cap > 0;
    const unsigned long long c = (unsigned long long)cap;
    if (f16 && col)
        hipLaunchKernelGGL((k_mesh<__half, true>), dim3(grid), dim3(kThreads), 0, s, view(g), n, triangles, colors, keys,
                           c, cnt);
    else if (f16)
        hipLaunchKernelGGL((k_mesh<__half, false>), dim3(grid), dim3(kThreads), 0, s, view(g), n, triangles, colors,
                           keys, c, cnt);
    else if (col)
        hipLaunchKernelGGL((k_mesh<float, true>), dim3(grid), dim3(kThreads), 0, s, view(g), n, triangles, colors, keys,
                           c, cnt);
    else
        hipLaunchKernelGGL((k_mesh<float, false>), dim3(grid), dim3(kThreads), 0, s, view(g), n, triangles, colors,
                           keys, c, cnt);
    unsigned long long h = 0;
    hipError_t e = hipGetLastError();
    if (e == hipSuccess)
        e = hipMemcpyAsync(&h, cnt, sizeof(h), hipMemcpyDeviceToHost, s);
    if (e == hipSuccess)
        e = hipStreamSynchronize(s);
    (void)hipFree(cnt);
    if (e != hipSuccess)
        return fail(TSDF_HIP_ERROR, std::string("mesh extraction: ") + hipGetErrorString(e));
    *n_triangles = h;
    return TSDF_OK;
}

}  // extern "C"
