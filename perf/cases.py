"""The work a user of this framework has it do, as measurable cases.

Each case is one pass of a scanning program (or of the differentiable
renderer) through the public entry points: the smallest camera, the ordinary
ones and the largest, fp32 and fp16 storage, with and without colour,
integrate and deintegrate, single calls and batches, forward and backward.
The maps are built from seeded synthetic frames (superscanner_amd.synth: the
analytic plain scene, the random room, the multi-room floor).

listed() names the cases, draw(rng) gives others of the same ranges,
prepare() makes the inputs and the map, run() makes one pass, work() counts
what a pass cannot do without, exact() gives the outputs in 64 bits from a
plain torch restatement (no code of this repository in it).
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from superscanner_amd import _lib, icp, synth
from superscanner_amd import diff_render as dr
from superscanner_amd.voxel_grid import GPUVoxelGrid

# scene -> camera and map parameters of its benchmark configuration, brick pool, hash buckets, spacing of
# the map's frames along the scene's trajectory, and the bricks that one frame touches (about)
SCENES = {
    "plain": dict(synth.PLAIN_SMALL, pool=1 << 17, n_buckets=1 << 20, touched=11000),
    "room": dict(synth.ROOM_LARGE, pool=1 << 17, n_buckets=1 << 22, touched=22000),
    "multi": dict(synth.FP16_LARGE, pool=1 << 21, n_buckets=1 << 23, touched=180000),
}
UPDATED = 0.47  # voxels of the touched bricks that a frame updates, about


def _case(name, kind, scene, H, W, frames, storage="f32", color=False, **more):
    return dict(name=name, kind=kind, scene=scene, H=H, W=W, frames=frames, storage=storage, color=color, **more)


def listed():
    return [
        # live scanning on the smallest camera: a frame fused and the model rendered for tracking, where launches
        # and latency count
        _case("scan_160x120", "scan", "plain", 120, 160, 8),
        # the same with colour at VGA
        _case("scan_color_640x480", "scan", "plain", 480, 640, 12, color=True),
        # the headline workload's step: a depth frame fused into the room and the model rendered
        _case("scan_848x480", "scan", "room", 480, 848, 30),
        # the largest camera on the finest map, half-precision storage
        _case("scan_f16_1280x720", "scan", "multi", 720, 1280, 20, storage="f16"),
        # a frame leaves the map (loop rejected), empty bricks are erased, the corrected frame comes back
        _case("forget_641x479", "forget", "room", 479, 641, 20),
        # the pose graph moved: 64 keyframes re-fused as one batch, the model rendered and the map saved
        _case("reintegrate_64", "reintegrate", "room", 480, 848, 64),
        # frame-to-frame registration, the reference's constants (10 iterations, 11 x 11 window)
        _case("icp_640x480", "icp", "room", 480, 640, 2, plane=False, iters=10),
        # its front end by itself: point maps, normal map, one point-to-plane association
        _case("frontend_848x480", "frontend", "room", 480, 848, 2, plane=True),
        # the differentiable renderer as a viewer: one VGA view with normals
        _case("render_640x480", "render", "plain", 480, 640, 12, views=1, h=480, w=640),
        # a training step through it: 16 views, gradients of the poses and of every voxel
        _case("train_16x320x240", "train", "plain", 480, 640, 12, views=16, h=240, w=320),
        # Gauss-Newton depth tracking of 16 views, 5 iterations
        _case("track_16x320x240", "track", "plain", 480, 640, 12, views=16, h=240, w=320, iters=5),
        # the scan's mesh at the end: sizes first, then vertices, normals and triangles
        _case("mesh_room", "mesh", "room", 480, 848, 30),
    ]


def draw(rng):
    """One more case of the ranges above."""
    def size(lo, hi):  # an image side pair of 3:4 to 9:16, spread over the logarithm, odd sizes too
        h = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        return h, int(round(h * rng.uniform(1.2, 1.77)))

    kind = rng.choice(["scan", "scan", "scan", "forget", "reintegrate", "icp", "frontend", "render", "train", "track",
                       "mesh"])
    if kind == "scan":
        scene = rng.choice(["plain", "room", "multi"])
        H, W = size(96, 720 if scene == "multi" else 480)
        return _draw(kind, scene, H, W, rng.randrange(6, 20),
                     "f16" if scene == "multi" else rng.choice(["f32", "f16"]),
                     scene != "multi" and rng.random() < 0.4)
    if kind in ("forget", "mesh"):
        H, W = size(160, 480)
        return _draw(kind, rng.choice(["plain", "room"]), H, W, rng.randrange(6, 24), rng.choice(["f32", "f16"]))
    if kind == "reintegrate":
        H, W = size(120, 480)
        return _draw(kind, "room", H, W, rng.randrange(3, 65), rng.choice(["f32", "f16"]), rng.random() < 0.3)
    if kind in ("icp", "frontend"):
        H, W = size(96, 480)
        more = dict(iters=rng.randrange(3, 11)) if kind == "icp" else {}
        return _draw(kind, rng.choice(["plain", "room"]), H, W, 2, plane=rng.random() < 0.5, **more)
    h, w = size(96, 480 if kind == "render" else 240)
    v = rng.randrange(1, 3 if kind == "render" else 15)
    more = dict(iters=rng.randrange(1, 6)) if kind == "track" else {}
    return _draw(kind, "plain", 480, 640, rng.randrange(6, 13), rng.choice(["f32", "f16"]), views=v, h=h, w=w, **more)


def _draw(*a, **k):
    c = _case("", *a, **k)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _scene(case, seed):
    """(prims, poses) of the case's frames (fp64, camera -> world)."""
    n, rng = case["frames"], np.random.default_rng(seed)
    if case["scene"] == "plain":
        a0, r, z = rng.uniform(0, 2 * math.pi), rng.uniform(1.3, 1.6), rng.uniform(0.8, 1.1)
        if case["kind"] in ("icp", "frontend"):  # consecutive frames
            ang = [a0 + 0.01 * k for k in range(n)]
        else:
            ang = [a0 + 2 * math.pi * k / n for k in range(n)]
        return synth.scene_plain_small(), [synth.look_at((r * math.cos(a), r * math.sin(a), z), (0, 0, 0.2))
                                           for a in ang]
    if case["scene"] == "room":
        prims, path = synth.scene_room(1 + seed % 1000), synth.traj_random_walk(600, seed=seed)
        if case["kind"] in ("icp", "frontend"):
            k0 = int(rng.integers(0, 500))
            return prims, [path[k0 + 3 * k] for k in range(n)]
        return prims, [path[(600 * k) // n] for k in range(n)]
    path = synth.traj_multiroom(2000, seed=seed)
    k0 = int(rng.integers(0, 2000))
    return synth.scene_multiroom(1 + seed % 1000), [path[(k0 + 15 * k) % 2000] for k in range(n)]


def _inputs(case, seed):
    cfg = dict(SCENES[case["scene"]])
    prims, poses = _scene(case, seed)
    H, W = case["H"], case["W"]
    cfg["intr"] = synth.scaled_intr(cfg, H, W)
    keep = np.random.default_rng(seed + 1).uniform(0.3, 1.0, len(poses)) if case["kind"] == "reintegrate" else None
    depth = torch.from_numpy(synth.frames(prims, poses, cfg, seed=seed % 100003, keep=keep, H=H, W=W).view(np.int16))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rgb = None
    if case["color"]:
        rgb = torch.randint(0, 256, (len(poses), H, W, 3), dtype=torch.uint8, device="cuda", generator=gen)
    return dict(cfg=cfg, poses=poses, E=[synth.pose_f32(T) for T in poses], depth=depth.cuda(), rgb=rgb,
                prims=prims)


def _views(case, seed, inp):
    """Render views near the map's poses, the depth a camera sees there (metres), and the intrinsics."""
    rng = np.random.default_rng(seed + 7)
    h, w = case["h"], case["w"]
    n = len(inp["poses"])
    true = [synth.perturb(inp["poses"][k % n], rng, 0.01, 1.0) for k in range(case["views"])]
    start = [synth.perturb(T, rng, 0.005, 0.3) for T in true]
    cfg = dict(SCENES[case["scene"]])
    cfg["intr"] = synth.scaled_intr(cfg, h, w)
    mm = synth.frames(inp["prims"], true, cfg, seed=seed % 9973, H=h, W=w)
    obs = torch.from_numpy((mm.astype(np.float32) / np.float32(1000.0))).cuda()
    return np.stack(start), obs, cfg["intr"]


def _new_poses(case, seed, inp):
    rng = np.random.default_rng(seed + 3)
    return [synth.pose_f32(synth.perturb(T, rng)) for T in inp["poses"]]


def _build(case, inp):
    cfg = inp["cfg"]
    g = GPUVoxelGrid(cfg["pool"] * 512, cfg["truncation"], cfg["voxel_length"], case["H"], case["W"],
                     n_buckets=cfg["n_buckets"], n_bricks=cfg["pool"], storage=case["storage"],
                     withColor=case["color"], max_weight=cfg["max_weight"])
    g.setIntrinsic(*cfg["intr"])
    for k, E in enumerate(inp["E"]):
        g.integrate(None if inp["rgb"] is None else inp["rgb"][k], inp["depth"][k], E)
    g.sync()
    return g


def _export(g):
    """The map's bricks and the permutation that puts them (ids depend on allocation races) in coordinate order."""
    e = g.export_bricks()
    c = e["coords"].long() + (1 << 20)
    return e, torch.argsort((c[:, 0] << 42) | (c[:, 1] << 21) | c[:, 2])


def prepare(case, seed):
    inp = _inputs(case, seed)
    s = dict(kind=case["kind"], at=0, **inp)
    if case["kind"] in ("icp", "frontend"):
        t = np.random.default_rng(seed + 5)
        s["tx"], s["ty"] = inp["poses"][0], synth.perturb(inp["poses"][1], t, 0.005, 0.2)
        s["type"] = icp.PointToPlane if case["plane"] else icp.PointToPoint
        s["iters"] = case.get("iters", 1)
        return s
    g = s["grid"] = _build(case, inp)
    if case["kind"] == "reintegrate":
        s["now"], s["next"] = inp["E"], _new_poses(case, seed, inp)
        s["keyframes"] = [inp["depth"][k] for k in range(len(inp["E"]))]
        s["colors"] = None if inp["rgb"] is None else [inp["rgb"][k] for k in range(len(inp["E"]))]
        g.reserve_batch(2 * len(inp["E"]))
        s["map"] = torch.zeros((2, 1 << 17, 512), dtype=torch.float32, device="cuda")  # the saved map, 0 beyond it
    elif case["kind"] in ("render", "train", "track"):
        s["T"], s["obs"], s["intr"] = _views(case, seed, inp)
        s["h"], s["w"], s["iters"] = case["h"], case["w"], case.get("iters", 0)
        if case["kind"] == "train":
            s["xi"] = torch.zeros((case["views"], 6), dtype=torch.float64, requires_grad=True)
            s["sdf"] = g.sdf_tensor().requires_grad_(True)
            s["order"] = _export(g)[1]
            s["grad"] = torch.zeros((1 << 16, 512), dtype=torch.float32, device="cuda")  # the map's spare rows are 0
    elif case["kind"] == "mesh":
        # the mesh's place: buffers with room to grow, 0 beyond it
        for name, n, dtype in (("vertices", 1 << 21, torch.float64), ("normals", 1 << 21, torch.float64)):
            s[name] = torch.zeros((n, 3), dtype=dtype, device="cuda")
        s["keys"] = torch.zeros(1 << 21, dtype=torch.int64, device="cuda")
        s["triangles"] = torch.zeros(1 << 22, dtype=torch.int64, device="cuda")
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _maps(s):
    g = s["grid"]
    out = dict(points=g.rayPcd, depth=g.rayDepth, flags=g.rayUB)
    if s["rgb"] is not None:
        out["colors"] = g.rayColorPcd
    return out


def run(s):
    kind = s["kind"]
    if kind in ("icp", "frontend"):
        intr, d = s["cfg"]["intr"], s["depth"]
        if kind == "icp":
            T, rmse, fit = icp.kokkosICP(d[0], d[1], s["tx"], s["ty"], intr, s["type"], n_it=s["iters"])
            return dict(T=T, rmse=np.float32(rmse), fitness=np.float32(fit))
        x, y = icp.CreatePcdFromDepthView(d[0], intr), icp.CreatePcdFromDepthView(d[1], intr)
        n = icp.CalculateNormalsFromPCDView(y)
        near = icp.associate(x, y, n, np.linalg.inv(s["ty"]) @ s["tx"], intr, s["type"])
        return dict(x=x, y=y, normals=n, nearest=near)
    g = s["grid"]
    if kind in ("scan", "forget"):
        k = s["at"] % len(s["E"])
        s["at"] += 1
        rgb = None if s["rgb"] is None else s["rgb"][k]
        out = {}
        if kind == "forget":
            g.deIntegrate(rgb, s["depth"][k], s["E"][k])
            out["removed"] = g.cleanMemory()
        g.integrate(rgb, s["depth"][k], s["E"][k])
        g.raycast(s["E"][k])
        return dict(out, **_maps(s))
    if kind == "reintegrate":
        g.reintegrate_batch(s["keyframes"], s["now"], s["next"], rgbs=s["colors"])
        s["now"], s["next"] = s["next"], s["now"]
        g.raycast(s["now"][0])
        e, order = _export(g)
        s["map"][0, :len(order)], s["map"][1, :len(order)] = e["sdf"][order], e["w"][order]
        return dict(_maps(s), map=s["map"])
    if kind == "render":
        depth, normals = dr.render(g, s["T"], s["h"], s["w"], s["intr"], normals=True)
        return dict(depth=depth, normals=normals)
    if kind == "train":
        depth = dr.RenderDepth.apply(s["xi"], s["sdf"], g, s["T"], s["h"], s["w"], s["intr"])
        r = depth - s["obs"]
        loss = torch.where((depth > 0) & (s["obs"] > 0) & (r.abs() < 0.1), r, 0.0).square().sum()
        gx, gs = torch.autograd.grad(loss, (s["xi"], s["sdf"]))
        s["grad"][:len(gs)] = gs[s["order"]]
        return dict(depth=depth.detach(), grad_xi=gx, grad_sdf=s["grad"])
    if kind == "track":
        T, hist = dr.track(g, s["obs"], s["T"], s["intr"], iters=s["iters"])
        return dict(T=T, rms=hist[-1]["rms"], count=hist[-1]["count"])
    return _mesh(g, s)


def _mesh(g, s):
    """tsdf_marching_cubes as a program calls it: the sizes, then the buffers.  Vertex and triangle order are free,
    so the mesh is put in the order of its vertex keys."""
    L, dev = g._L, g.device
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    nv, nt = C.c_uint64(0), C.c_uint64(0)
    _lib.check(L.tsdf_marching_cubes(g._h, None, None, None, None, None, 0, 0, C.byref(nv), C.byref(nt), stream),
               "tsdf_marching_cubes")
    v = torch.empty((nv.value, 3), dtype=torch.float64, device=dev)
    n = torch.empty((nv.value, 3), dtype=torch.float64, device=dev)
    f = torch.empty((nt.value, 3), dtype=torch.int32, device=dev)
    k = torch.empty((nv.value,), dtype=torch.int64, device=dev)
    p = [C.c_void_p(t.data_ptr()) for t in (v, n, f, k)]
    _lib.check(L.tsdf_marching_cubes(g._h, p[0], None, p[1], p[2], p[3], nv.value, nt.value, C.byref(nv),
                                     C.byref(nt), stream), "tsdf_marching_cubes")
    keys, order = torch.sort(k)
    rank = torch.empty_like(order)
    rank[order] = torch.arange(len(order), device=dev)
    t = rank[f.long()]
    s["vertices"][:len(v)], s["normals"][:len(v)], s["keys"][:len(v)] = v[order], n[order], keys
    s["triangles"][:len(t)] = torch.sort((t[:, 0] << 42) | (t[:, 1] << 21) | t[:, 2])[0]
    return {k: s[k] for k in ("vertices", "normals", "keys", "triangles")}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    cfg = SCENES[case["scene"]]
    px = case["H"] * case["W"]
    kind = case["kind"]
    sv = (4 if case["storage"] == "f16" else 8) + (12 if case["color"] else 0)  # bytes of a voxel
    nt = cfg["touched"]
    fuse = dict(bytes=px * (5 if case["color"] else 2) + nt * 512 * sv * (1 + UPDATED) + nt * 8,
                flops=nt * 512 * 35)
    ray = dict(bytes=px * (17 + 12) + px * 8 * sv, flops=px * 14 * 40)
    if kind in ("icp", "frontend"):
        it = case.get("iters", 1)
        return dict(bytes=px * (4 + 36) + it * px * (36 + (12 if case["plane"] else 0)), flops=it * px * 100 * 9)
    if kind in ("scan", "forget", "reintegrate"):
        n = {"scan": 1, "forget": 2, "reintegrate": 2 * case["frames"]}[kind]
        # a batch reads and writes each brick of the map once
        once = fuse["bytes"] if kind == "reintegrate" else n * fuse["bytes"]
        extra = px * (5 if case["color"] else 2) * case["frames"] if kind == "reintegrate" else 0
        saved = 2 * nt * 512 * (sv + 8) if kind == "reintegrate" else 0
        return dict(bytes=once + extra + saved + ray["bytes"], flops=n * fuse["flops"] + ray["flops"])
    if kind == "mesh":
        m = 2 * nt  # bricks of the map
        return dict(bytes=m * 512 * sv + m * 32 * (24 + 24 + 8) + m * 62 * 12, flops=m * 512 * 20)
    rays = case["views"] * case["h"] * case["w"]
    if kind == "render":
        return dict(bytes=rays * (16 + 8 * sv), flops=rays * 30 * 60)
    if kind == "train":
        return dict(bytes=rays * (4 + 8 * sv) + rays * (8 + 8 * sv + 32) + 4 * nt * 512, flops=rays * 30 * 60)
    return dict(bytes=case["iters"] * rays * (4 + 8 * sv), flops=case["iters"] * rays * (30 * 60 + 60))


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
F = torch.float64


def _t(a):
    return torch.as_tensor(np.asarray(a, np.float64), dtype=F, device="cuda")


def _pack(b):
    b = b + (1 << 20)
    return (b[..., 0] << 42) | (b[..., 1] << 21) | b[..., 2]


def _unpack(k):
    return torch.stack([(k >> 42) & 0x1FFFFF, (k >> 21) & 0x1FFFFF, k & 0x1FFFFF], -1) - (1 << 20)


def _index(a, d):  # the reference's block / voxel index: (int)(a / d), one less below zero
    q = a / d
    return torch.where(a >= 0, q, q - 1).trunc().long()


class _Map:
    """The voxel-hashed TSDF with its bricks in key order, 64-bit values."""

    def __init__(self, case, cfg):
        self.vl, self.dt = float(np.float32(cfg["voxel_length"])), float(np.float32(cfg["truncation"]))
        self.vbl, self.wmax = 8 * self.vl, cfg["max_weight"]
        self.H, self.W = case["H"], case["W"]
        self.cam = _camera(cfg["intr"], self.H)
        self.color = case["color"]
        self.keys = torch.empty(0, dtype=torch.int64, device="cuda")
        self.s, self.w = (torch.empty((0, 512), dtype=F, device="cuda") for _ in range(2))
        self.c = torch.empty((0, 512, 3), dtype=F, device="cuda") if self.color else None

    def _keep(self, keys):
        """The map over `keys` (sorted), bricks it had keep their values."""
        at, had = _find(self.keys, keys) if len(self.keys) else (torch.zeros_like(keys), torch.zeros_like(keys) > 0)
        for name in ("s", "w", "c"):
            v = getattr(self, name)
            if v is not None:
                new = torch.zeros((len(keys),) + v.shape[1:], dtype=F, device="cuda")
                new[had] = v[at[had]]
                setattr(self, name, new)
        self.keys = keys

    def clean(self):
        n = len(self.keys)
        self._keep(self.keys[(self.w != 0).any(1)])
        return n - len(self.keys)

    def op(self, depth, rgb, E, sign):
        E = _t(E)
        R, t = E[:3, :3], E[:3, 3]
        Ez = R[:, 2] / R[:, 2].norm()
        cam = _points(depth, self.cam)
        pw = cam @ R.T + t
        ok = (cam[..., 2] > float(np.float32(0.2))).reshape(-1)
        p = pw.reshape(-1, 3)[ok]
        lo, hi = _index(p - self.dt, self.vbl), _index(p + self.dt, self.vbl)
        keys = []
        ext = (hi - lo).amax(0).tolist() if len(p) else [-1, -1, -1]
        for x in range(ext[0] + 1):
            for y in range(ext[1] + 1):
                for z in range(ext[2] + 1):
                    b = lo + torch.tensor([x, y, z], device="cuda")
                    keys.append(torch.unique(_pack(b[(b <= hi).all(1)])))
        mine = torch.unique(torch.cat(keys)) if keys else self.keys[:0]
        self._keep(torch.unique(torch.cat([self.keys, mine])))
        fx, fy, ci, cj = self.cam
        v = torch.arange(512, device="cuda")
        off = (torch.stack([v & 7, (v >> 3) & 7, v >> 6], -1).to(F) + 0.5) * self.vl
        ids = _find(self.keys, mine)[0]
        for a in range(0, len(mine), 16384):
            i = ids[a:a + 16384]
            vm = _unpack(mine[a:a + 16384]).to(F)[:, None] * self.vbl + off
            c = (vm - t) @ R
            row, col = (c[..., 1] * fy / c[..., 2] + ci).trunc(), (c[..., 0] * fx / c[..., 2] + cj).trunc()
            inside = (row >= 0) & (row < self.H) & (col >= 0) & (col < self.W)
            pix = torch.where(inside, row * self.W + col, 0.0).long()
            sdf = ((pw.reshape(-1, 3)[pix] - vm) * Ez).sum(-1)
            upd = inside & ok[pix] & (sdf.abs() < self.dt)
            s, w = self.s[i], self.w[i]
            d = w + sign
            zero = (w == 1) & (sign < 0)
            dd = torch.where(d == 0, 1.0, d)
            self.s[i] = torch.where(upd, torch.where(zero, 0.0, (s * w + sign * sdf) / dd), s)
            if self.color:
                q = (self.c[i] * w[..., None] + sign * rgb.reshape(-1, 3)[pix].to(F)) / dd[..., None]
                self.c[i] = torch.where(upd[..., None], torch.where(zero[..., None], 0.0, q), self.c[i])
            cap = (w >= self.wmax) if self.wmax > 0 and sign > 0 else torch.zeros_like(zero)
            self.w[i] = torch.where(upd, torch.where(zero, 0.0, torch.where(cap, float(self.wmax), d)), w)

    def raycast(self, E):
        E = _t(E)
        R, o = E[:3, :3], E[:3, 3]
        vl, vbl, dt, far = self.vl, self.vbl, self.dt, 10.0
        n = _rays(self.H, self.W, self.cam).reshape(-1, 3)
        n = n / n.norm(dim=1, keepdim=True)
        N = len(n)
        dirs = n @ R.T
        points, colors = torch.zeros((N, 3), dtype=F, device="cuda"), torch.zeros((N, 3), dtype=F, device="cuda")
        hit = torch.zeros(N, dtype=torch.bool, device="cuda")
        at = torch.arange(N, device="cuda")  # rays under way, and their state
        rv, l = o + 0.1 * dirs, torch.full((N,), 0.1, dtype=F, device="cuda")
        phase = torch.zeros(N, dtype=torch.long, device="cuda")  # 0 skip, 1 re-advance, 2 walk
        steps, seen = torch.zeros_like(phase), torch.zeros_like(hit)
        blk = torch.zeros((N, 3), dtype=torch.long, device="cuda")
        while len(at):
            d = dirs[at]
            b = _index(rv, vbl)
            id_, found = _find(self.keys, _pack(b))
            left = (phase == 2) & (b != blk).any(1)  # the walk left its block: look up again
            ph = torch.where(left, 0, phase)
            steps = torch.where(left, 0, steps)
            vox = _index(rv - vbl * b.to(F), vl)
            bad = ((vox < 0) | (vox > 7)).any(1)
            vi = (vox[:, 0] + 8 * vox[:, 1] + 64 * vox[:, 2]).clamp(0, 511)
            s, w = self.s[id_, vi], self.w[id_, vi]
            walk = (ph == 2) & ~bad
            front = walk & (w > 0) & ~(s > 0)
            cross = torch.nonzero(front & seen)[:, 0]
            if len(cross):
                m, dc = at[cross], d[cross]
                r2 = rv[cross] - vl * dc
                b2 = _index(r2, vbl)
                i2, f2 = _find(self.keys, _pack(b2))
                x2 = _index(r2 - vbl * b2.to(F), vl)
                fine = f2 & ((x2 >= 0) & (x2 <= 7)).all(1)
                v2 = (x2[:, 0] + 8 * x2[:, 1] + 64 * x2[:, 2]).clamp(0, 511)
                s1, w1, s2, w2 = s[cross], w[cross], self.s[i2, v2], self.w[i2, v2]
                f = (w2 * s2 / vl + w1 * (1 - s1 / vl)) / (w1 + w2)
                m1 = b[cross].to(F) * vbl + (vox[cross].to(F) + 0.5) * vl
                m2 = b2.to(F) * vbl + (x2.to(F) + 0.5) * vl
                p = m2 + f[:, None] * (m1 - m2)
                p = r2 + (((p - r2) * dc).sum(1))[:, None] * dc
                points[m[fine]], hit[m[fine]] = p[fine], True
                if self.color:
                    c = (0.5 * self.c[i2, v2] + 0.5 * self.c[id_[cross], vi[cross]]) / 255.0
                    colors[m[fine]] = c[fine]
            stop = front | ((ph == 2) & bad)
            seen = torch.where(walk, w > 0, seen)
            back = (ph == 0) & found & (steps > 0)
            go = torch.where(ph == 2, vl, torch.where(ph == 1, torch.where(found, 0.0, dt),
                                                     torch.where(found, torch.where(back, -(vbl - dt), 0.0), vbl)))
            nph = torch.where(back, 1, torch.where(found, 2, ph))
            blk = torch.where((nph == 2)[:, None], b, blk)
            steps = steps + ((ph == 0) & ~found).long()
            rv, l = rv + go[:, None] * d, l + go
            on = torch.nonzero(~stop & (l < far))[:, 0]
            at, rv, l, phase, steps, seen, blk = (v[on] for v in (at, rv, l, nph, steps, seen, blk))
        depth = torch.where(hit, ((points - o) @ R[:, 2]), 0.0)
        sh = (self.H, self.W)
        return points.reshape(sh + (3,)), depth.reshape(sh), colors.reshape(sh + (3,))

    # the trilinear field of the differentiable render at points p [n, 3]: (defined, phi, gradient, voxels, weights)
    def field(self, p):
        u = p / self.vl - 0.5
        k = u.floor()
        fr, k = u - k, k.long()
        phi, ok = torch.zeros(len(p), dtype=F, device="cuda"), torch.ones(len(p), dtype=torch.bool, device="cuda")
        grad = torch.zeros((len(p), 3), dtype=F, device="cuda")
        idx, wts = [], []
        for c in range(8):
            a = torch.tensor([c & 1, (c >> 1) & 1, c >> 2], device="cuda")
            v = k + a
            i, found = _find(self.keys, _pack(v >> 3))
            x = v & 7
            vi = x[:, 0] + 8 * x[:, 1] + 64 * x[:, 2]
            ok &= found & (self.w[i, vi] > 0)
            q = torch.where(a > 0, fr, 1 - fr)
            sg = torch.where(a > 0, 1.0, -1.0).to(F)
            val = self.s[i, vi]
            wt = q.prod(1)
            phi += wt * val
            grad += torch.stack([sg[0] * q[:, 1] * q[:, 2], q[:, 0] * sg[1] * q[:, 2], q[:, 0] * q[:, 1] * sg[2]],
                                1) * val[:, None] / self.vl
            idx.append(i * 512 + vi)
            wts.append(wt)
        return ok, phi, grad, torch.stack(idx, 1), torch.stack(wts, 1)

    def render(self, T, h, w, intr):
        """Depth [views * h * w], and at the hits: which, points, gradients, slopes, voxels and weights."""
        E = _t(np.asarray(T).astype(np.float32))
        o = E[:, None, :3, 3].expand(-1, h * w, -1).reshape(-1, 3)
        d = torch.cat([_rays(h, w, _camera(intr, h)).reshape(-1, 3) @ e[:3, :3].T for e in E])
        dn = d.norm(dim=1)
        N, near, far = len(d), float(np.float32(0.2)), 10.0
        at = torch.arange(N, device="cuda")
        lam = torch.full((N,), near, dtype=F, device="cuda")
        pl, pp, pv = torch.zeros_like(lam), torch.zeros_like(lam), torch.zeros(N, dtype=torch.bool, device="cuda")
        A, B, got = torch.zeros_like(lam), torch.zeros_like(lam), torch.zeros_like(pv)
        while len(at):
            r = d[at]
            p = o[at] + lam[:, None] * r
            ok, phi = self.field(p)[:2]
            x = ok & pv & (pp > 0) & (phi <= 0)
            A[at[x]], B[at[x]], got[at[x]] = pl[x], lam[x], True
            b = (p / self.vbl).floor().long()
            found = _find(self.keys, _pack(b))[1]
            edge = torch.where(r > 0, (b + 1).to(F) * self.vbl - o[at], b.to(F) * self.vbl - o[at]) / r
            te = torch.where(r == 0, math.inf, edge).amin(1)
            eps = 1e-3 * self.vl / dn[at]
            st = torch.where(ok, torch.clamp(0.5 * phi.abs(), min=0.5 * self.vl) / dn[at],
                             torch.where(found, 0.5 * self.vl / dn[at], torch.maximum(te - lam + eps, eps)))
            pl, pp, pv, lam = lam, phi, ok, lam + st
            on = torch.nonzero(~x & (lam < far))[:, 0]
            at, lam, pl, pp, pv = at[on], lam[on], pl[on], pp[on], pv[on]
        m = torch.nonzero(got)[:, 0]
        a, b = A[m], B[m]
        for _ in range(52):
            x = 0.5 * (a + b)
            phi = self.field(o[m] + x[:, None] * d[m])[1]
            a, b = torch.where(phi > 0, x, a), torch.where(phi > 0, b, x)
        x = 0.5 * (a + b)
        p = o[m] + x[:, None] * d[m]
        ok, _, grad, idx, wts = self.field(p)
        s = (grad * d[m]).sum(1)
        ok &= s < -0.05 * grad.norm(dim=1) * dn[m]
        depth = torch.zeros(N, dtype=F, device="cuda")
        depth[m[ok]] = x[ok]
        return depth, m[ok], p[ok], grad[ok], s[ok], idx[ok], wts[ok]


def _find(keys, q):
    i = torch.searchsorted(keys, q).clamp(max=len(keys) - 1)
    return i, keys[i] == q


def _camera(intr, H):
    fx, fy, cx, cy = (float(np.float32(v)) for v in intr)
    return fx, fy, float(np.float32(H) - np.float32(cy)), cx


def _rays(H, W, cam):
    fx, fy, ci, cj = cam
    i, j = torch.meshgrid(torch.arange(H, dtype=F, device="cuda"), torch.arange(W, dtype=F, device="cuda"),
                          indexing="ij")
    return torch.stack([(j - cj) / fx, (i - ci) / fy, torch.ones_like(i)], -1)


def _points(depth, cam):
    d = (depth.long() & 0xFFFF).to(F) / 1000.0
    return _rays(*depth.shape, cam) * d[..., None]


def _normals(p):
    n = torch.zeros_like(p)
    n[..., 2] = 1.0
    c, dn, up, rt, lf = p[1:-1, 1:-1], p[2:, 1:-1], p[:-2, 1:-1], p[1:-1, 2:], p[1:-1, :-2]
    x = lambda a, b: torch.linalg.cross(a - c, b - c)  # noqa: E731
    s = x(dn, rt) + x(lf, dn) + x(rt, up) + x(up, lf)
    ok = (c[..., 2] != 0) & (dn[..., 2] != 0) & (up[..., 2] != 0) & (rt[..., 2] != 0) & (lf[..., 2] != 0)
    n[1:-1, 1:-1] = torch.where(ok[..., None], s / s.norm(dim=-1, keepdim=True), n[1:-1, 1:-1])
    return n


def _nearest(x, y, n, T, cam, plane, ns=5, most=float(np.float32(0.075))):
    H, W = x.shape[:2]
    fx, fy, ci, cj = cam
    px = x @ T[:3, :3].T + T[:3, 3]
    z = torch.where(x[..., 2] != 0, px[..., 2], 1.0)
    r, c = (px[..., 1] * fy / z + ci).trunc().long(), (px[..., 0] * fx / z + cj).trunc().long()
    act = (x[..., 2] != 0) & (r > ns) & (r < H - ns) & (c > ns) & (c < W - ns)
    best = torch.full((H, W), 1e6, dtype=F, device="cuda")
    out = torch.zeros_like(x)
    for a in range(-ns, ns):
        for b in range(-ns, ns):
            q = torch.where(act, (r + a) * W + c + b, 0)
            py, nv = y.reshape(-1, 3)[q], n.reshape(-1, 3)[q]
            if plane:
                d = ((py - px) * nv).sum(-1)
                dist, to, use = d.abs(), px + d[..., None] * nv, nv[..., 0] != 0
            else:
                dist, to, use = (py - px).norm(dim=-1), py, act
            new = act & use & (py[..., 2] != 0) & (dist < best) & (dist < most)
            best = torch.where(new, dist, best)
            out = torch.where(new[..., None], to, out)
    return out


def _icp(x, y, n, T, cam, plane, iters):
    low, best, fit = 1e6, torch.eye(4, dtype=F, device="cuda"), 0.0
    for _ in range(iters):
        near = _nearest(x, y, n, T, cam, plane)
        m = near[..., 2] != 0
        if not m.any():
            break
        a, b = x[m], near[m]
        ca, cb = a.mean(0), b.mean(0)
        rmse = float(((b - (a @ T[:3, :3].T + T[:3, 3])) ** 2).sum(1).mean().sqrt())
        fit = max(fit, float(m.sum()) / float((x[..., 2] != 0).sum()))
        U, _, Vt = torch.linalg.svd((a - ca).T @ (b - cb))
        T = torch.eye(4, dtype=F, device="cuda")
        T[:3, :3] = Vt.T @ U.T
        T[:3, 3] = cb - T[:3, :3] @ ca
        if rmse < low:
            low, best = rmse, T
    return best, low, fit


def _jacobian(p, grad, s):  # d depth / d xi of the left perturbation
    return torch.cat([-grad, -torch.linalg.cross(p, grad)], 1) / s[:, None]


def exact(case, seed):
    kind = case["kind"]
    if kind == "mesh":
        return None
    inp = _inputs(case, seed)
    if kind in ("icp", "frontend"):
        cam = _camera(inp["cfg"]["intr"], case["H"])
        ty = synth.perturb(inp["poses"][1], np.random.default_rng(seed + 5), 0.005, 0.2)
        T = _t(np.linalg.inv(ty) @ inp["poses"][0])
        x, y = _points(inp["depth"][0], cam), _points(inp["depth"][1], cam)
        n = _normals(y)
        if kind == "icp":
            T, rmse, fit = _icp(x, y, n, T, cam, case["plane"], case["iters"])
            return dict(T=T, rmse=rmse, fitness=fit)
        return dict(x=x, y=y, normals=n, nearest=_nearest(x, y, n, T, cam, case["plane"]))
    m = _Map(case, inp["cfg"])
    rgb = lambda k: None if inp["rgb"] is None else inp["rgb"][k]  # noqa: E731
    for k, E in enumerate(inp["E"]):
        m.op(inp["depth"][k], rgb(k), E, 1)
    if kind in ("scan", "forget", "reintegrate"):
        E = inp["E"][0]
        if kind == "forget":
            m.op(inp["depth"][0], rgb(0), E, -1)
            m.clean()
        if kind == "reintegrate":
            new = _new_poses(case, seed, inp)
            for k, E in enumerate(inp["E"]):
                m.op(inp["depth"][k], rgb(k), E, -1)
                m.op(inp["depth"][k], rgb(k), new[k], 1)
            E = new[0]
        else:
            m.op(inp["depth"][0], rgb(0), E, 1)
        points, depth, colors = m.raycast(E)
        out = dict(points=points, depth=depth, flags=None, map=None)
        if case["color"]:
            out["colors"] = colors
        return out
    T, obs, intr = _views(case, seed, inp)
    h, w, n = case["h"], case["w"], case["views"]
    for it in range(case.get("iters", 1)):
        depth, at, p, grad, s, idx, wts = m.render(T, h, w, intr)
        view, dobs = at // (h * w), obs.reshape(-1)[at].to(F)
        r, J = depth[at] - dobs, _jacobian(p, grad, s)
        use = (dobs > 0) & (r.abs() < 0.1)
        if kind != "track":
            break
        rms, count, T = [], [], np.array(T)
        for v in range(n):
            Jv, rv = J[use & (view == v)], r[use & (view == v)]
            rms.append(float((rv * rv).mean().sqrt()))
            count.append(float(len(rv)))
            T[v] = _exp(torch.linalg.solve(Jv.T @ Jv, -Jv.T @ rv).cpu().numpy()) @ T[v]
    if kind == "track":
        return dict(T=T, rms=np.array(rms), count=np.array(count))
    depth = depth.reshape(n, h, w)
    if kind == "render":
        normals = torch.zeros((n * h * w, 3), dtype=F, device="cuda")
        normals[at] = grad / grad.norm(dim=1, keepdim=True)
        return dict(depth=depth, normals=normals.reshape(n, h, w, 3))
    gd = torch.where(use, 2 * r, 0.0)
    gx = torch.zeros((n, 6), dtype=F, device="cuda").index_add_(0, view, J * gd[:, None])
    gs = torch.zeros((1 << 16) * 512, dtype=F, device="cuda")
    gs.index_add_(0, idx.reshape(-1), (-wts / s[:, None] * gd[:, None]).reshape(-1))
    return dict(depth=depth, grad_xi=gx, grad_sdf=gs.reshape(-1, 512))


def _exp(xi):
    """exp of a twist (v, w) as a 4x4 matrix."""
    K = np.zeros((4, 4))
    K[:3, :3] = [[0, -xi[5], xi[4]], [xi[5], 0, -xi[3]], [-xi[4], xi[3], 0]]
    K[:3, 3] = xi[:3]
    return torch.linalg.matrix_exp(torch.from_numpy(K)).numpy()
