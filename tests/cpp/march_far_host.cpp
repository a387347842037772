// Host build of the raycast march with its far bound and its deferral, for
// tests/test_march_far_host.py.  The per-lane march runs with both tile bounds
// and a budget; a ray it defers is finished from the saved state alone by the
// reference's loops written out one lookup at a time (GPUVoxelGrid.cpp:589-706),
// so a wrong position, length, count or phase in the state shows.
#include "march_host.cpp"

namespace {

// The far map of one raycast, as k_ray_bounds builds it (grow and the clip
// depth as the host side of tsdf_raycast computes them).
std::vector<unsigned long long> far_map(const HostRaycast& h, int n, const int32_t* coords, int fx, int fy)
{
    const GridView& g = h.g;
    const double dm = g.dmax, vbl = g.vbl, R0 = 0.0;
    const double n_upd = 4.0 * (dm + vbl) / std::fmin((double)g.vl, (double)g.trunc) + 64.0;
    double tmax = R0;
    for (int a = 0; a < 3; ++a)
        tmax = std::fmax(tmax, std::fabs((double)h.P.E[4 * a + 3]));
    auto spacing = [](double x) { return std::ldexp(1.0, std::ilogb(x) - 23); };
    const double R = tmax + dm + vbl + 1.0, s3 = std::sqrt(3.0);
    const float grow = (float)(s3 * n_upd * spacing(R) / 2.0 + n_upd * spacing(dm + vbl) / 2.0 +
                               s3 * n_upd * spacing(vbl) / 2.0 + s3 * dm * spacing(R) + 8.0 * spacing(R) + 1e-4);
    const double ex = std::fmax(std::fabs(g.cam.cj / g.cam.fx), std::fabs((g.W - 1.0 - g.cam.cj) / g.cam.fx));
    const double ey = std::fmax(std::fabs(g.cam.ci / g.cam.fy), std::fabs((g.H - 1.0 - g.cam.ci) / g.cam.fy));
    const float z_lo = (float)(0.1 / std::sqrt(1.0 + ex * ex + ey * ey) * (1.0 - 1e-4) - grow);
    std::vector<unsigned long long> zf((size_t)fx * fy, 0ull);
    for (int b = 0; b < n; ++b) {
        const int* c = coords + 3 * b;
        float zmin, zmax;
        int r0, r1, c0, c1;
        if (!brick_span(c[0], c[1], c[2], g.vbl, h.P, g.cam, g.H, g.W, grow, z_lo, zmin, zmax, r0, r1, c0, c1))
            continue;
        const unsigned long long v = tb_pack_far(1u, zmax);
        for (int y = r0 / kTbFarTile; y <= r1 / kTbFarTile; ++y)
            for (int x = c0 / kTbFarTile; x <= c1 / kTbFarTile; ++x)
                zf[(size_t)y * fx + x] = std::max(zf[(size_t)y * fx + x], v);
    }
    return zf;
}

struct Plain {  // a ray at its lookups
    const GridView& g;
    const RayParams& rp;
    f3 rv, dir;
    float l;
    RayResult out;
    int look()
    {
        int x, y, z;
        vb3(rv, rp, x, y, z);
        ++out.probes;
        return find_brick(g, x, y, z);
    }
    void step(float d)
    {
        rv = {rv.x + d * dir.x, rv.y + d * dir.y, rv.z + d * dir.z};
        l += d;
    }
    // the lookups of a run from rv on; taken: that at rv was made and missed
    int run(float d, bool taken, int& steps)
    {
        int id = taken ? -1 : look();
        while (id < 0 && l < rp.dmax) {
            step(d);
            ++steps;
            id = look();
        }
        return id;
    }
};

// The rest of a deferred ray; false when the lookup it carries is not that of its position.
bool finish(const GridView& g, const Pose& P, const RayParams& rp, const RayState& st, RayResult& res)
{
    const int i = (int)(st.pix / (uint32_t)rp.W), j = (int)(st.pix % (uint32_t)rp.W);
    Plain m{g, rp, {st.rx, st.ry, st.rz}, {}, st.l, {}};
    f3 n, rv0;
    ray_setup(g, P, i, j, n, rv0, m.dir);
    m.out.samples = st.samples;
    m.out.probes = st.probes;
    bool Lp = (st.flags & kRayLp) != 0, skip = (st.flags & kRaySkip) != 0, adv = (st.flags & kRayAdvance) != 0;
    if (st.flags & kRayPre) {
        int x, y, z;
        vb3(m.rv, rp, x, y, z);
        if (skip || adv || st.pre_key != prime_hash(x, y, z) || st.pre_bk != (mix32(st.pre_key) & g.mask) ||
            st.pre_slot != g.slots[st.pre_bk])
            return false;
    }
    while (m.l < rp.dmax) {
        int steps = skip ? 1 : 0, again = 0, id = -1;
        if (!adv) {
            id = m.run(rp.vbl, skip, steps);
            if (!(m.l < rp.dmax))
                break;
            if (steps > 0) {
                const float back = rp.back;
                m.rv = {m.rv.x - back * m.dir.x, m.rv.y - back * m.dir.y, m.rv.z - back * m.dir.z};
                m.l -= back;
            }
        }
        if (adv || steps > 0)
            id = m.run(rp.dt, adv && !(st.flags & kRayFirst), again);
        skip = adv = false;
        if (!(m.l < rp.dmax))
            break;
        int bx, by, bz;
        vb3(m.rv, rp, bx, by, bz);
        for (;;) {
            int qx, qy, qz, vx, vy, vz;
            vb3(m.rv, rp, qx, qy, qz);
            if (!(m.l < rp.dmax) || qx != bx || qy != by || qz != bz)
                break;
            vin3(m.rv, bx, by, bz, rp, vx, vy, vz);
            if (!vin_ok(vx, vy, vz)) {
                m.out.code = -kRayUbVoxelIndex;
                res = m.out;
                return true;
            }
            const int v = vx + kVPE * vy + kVPE * kVPE * vz;
            float s, w;
            ld_pair((const float*)g.payload + (size_t)id * (2 * kVPB), v, s, w);
            ++m.out.samples;
            if (w > 0 && !(s > 0)) {
                if (Lp)
                    crossing<float, false, false>(g, rp, Footprint{}, m.rv, m.l, m.dir, bx, by, bz, id, s, w, v, m.out);
                res = m.out;
                return true;
            }
            Lp = w > 0;
            const f3 d = {rp.vl * m.dir.x, rp.vl * m.dir.y, rp.vl * m.dir.z};
            m.rv = add3(m.rv, d);
            m.l += rp.vl;
        }
    }
    res = m.out;
    return true;
}

}  // namespace

// counts: [0] samples, [1] probes, [2] lookups loaded with both bounds, [3] with the near one alone, [4] deferred
// rays, [5] of them inside a skip, [6] inside a re-advance, [7] with a lookup loaded ahead.
extern "C" int march_far_host(int H, int W, float fx, float fy, float cx, float cy, float vl, float trunc, float dmax,
                              int n, const int64_t* keys, const int32_t* coords, const float* sdf, const float* w,
                              uint32_t n_buckets, const float* E, int budget, float* points, float* depth, uint8_t* ub,
                              uint64_t* counts)
{
    HostRaycast h;
    if (build(h, H, W, fx, fy, cx, cy, vl, trunc, dmax, n, keys, coords, sdf, w, n_buckets, 2, E) || !h.rp.use_tb)
        return 1;
    const int tfx = (W + kTbFarTile - 1) / kTbFarTile, tfy = (H + kTbFarTile - 1) / kTbFarTile;
    const std::vector<unsigned long long> zf = far_map(h, n, coords, tfx, tfy);
    Footprint fp;
    std::memset(&fp, 0, sizeof(fp));
    uint64_t loaded = 0;
    HostTrace hook = {[](void* c, uint32_t) { ++*(uint64_t*)c; }, [](void*, int, int) {}, &loaded};
    for (int k = 0; k < 8; ++k)
        counts[k] = 0;
    for (int i = 0; i < H; ++i)
        for (int j = 0; j < W; ++j) {
            const float zt = h.tile_depth(i, j);
            const float z = tb_far(zf[(size_t)(i / kTbFarTile) * tfx + j / kTbFarTile], 1u);
            RayState st;
            std::memset(&st, 0, sizeof(st));
            RayResult r = march<float, false, false>(h.g, h.P, h.rp, i, j, fp, zt, budget, &st, z);
            if (r.code == kRayDeferred) {
                ++counts[4];
                counts[5] += (st.flags & kRaySkip) ? 1 : 0;
                counts[6] += (st.flags & kRayAdvance) ? 1 : 0;
                counts[7] += (st.flags & kRayPre) ? 1 : 0;
                if (st.zt != zt || st.zf != z || !finish(h.g, h.P, h.rp, st, r))
                    return 2;
            }
            const size_t o = (size_t)i * W + j;
            points[o * 3 + 0] = r.p.x;
            points[o * 3 + 1] = r.p.y;
            points[o * 3 + 2] = r.p.z;
            depth[o] = r.code == 1 ? (r.p.x * h.P.Ei[8] + r.p.y * h.P.Ei[9] + r.p.z * h.P.Ei[10] + h.P.Ei[11]) : 0.0f;
            ub[o] = (uint8_t)(r.code < 0 ? -r.code : 0);
            counts[0] += r.samples;
            counts[1] += r.probes;
            host_trace() = &hook;
            for (int k = 0; k < 2; ++k) {
                loaded = 0;
                march<float, false, true>(h.g, h.P, h.rp, i, j, fp, zt, 0, nullptr, k ? -1.0f : z);
                counts[2 + k] += loaded;
            }
            host_trace() = nullptr;
        }
    return 0;
}

extern "C" int budget_of(int budget, int bounds, int W, int H, int n_cu)
{
    return raycast_budget(budget, bounds != 0, W, H, n_cu);
}
