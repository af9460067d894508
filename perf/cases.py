"""Workloads of the reconstruction path, for timing and for comparing outputs.

listed() gives fixed cases, draw() more of the same ranges, prepare() what a
program holds before the call (scene, frames, volume), run() one pass through
the package's public entry points with its outputs, work() the bytes and
operations a pass cannot do without and exact() the outputs in 64 bits where
they are plain arithmetic on the inputs.

Scenes are the package's seeded synthetic ones: "room" (a camera turning inside
a room, 20 poses around it) and "desk" (a slowly moving camera over eight
primitives, 2 % holes).  Voxel sizes, pool sizes and intrinsics follow
meshhashing_amd.configs: truncation is four voxels throughout.
"""
from __future__ import annotations

import math
from dataclasses import replace

import numpy as np
import torch

from meshhashing_amd import _capi as A
from meshhashing_amd.configs import C1, C2, C3, c4_scenes
from meshhashing_amd.engine import Batch, MainEngine, Volume, synth_color, synth_depth, synth_pose

# voxel size in mm -> (buckets, block pool, vertex pool), as the configurations size them; a
# probabilistic scan with 10 % outliers allocates several times the surface's blocks
POOLS = {5: (1 << 20, 1 << 19, 8 << 20), 10: (1 << 18, 1 << 17, 2 << 20), 20: (1 << 17, 1 << 15, 1 << 20),
         40: (1 << 16, 1 << 13, 1 << 18)}


def listed():
    return [
        # a coarse preview of a finished model, the smallest call: one small image
        {"name": "render_160x120_4cm", "kind": "render", "scene": "room", "w": 160, "h": 120, "mm": 40, "frames": 10},
        # viewing the full-resolution model from a new pose
        {"name": "render_640x480_5mm", "kind": "render", "scene": "desk", "w": 640, "h": 480, "mm": 5, "frames": 12},
        # a large still of it, of no particular size
        {"name": "render_1237x931_5mm", "kind": "render", "scene": "room", "w": 1237, "h": 931, "mm": 5, "frames": 8},
        # live scanning stage by stage from host frames, with meshing and block recycling, and the view of it
        {"name": "live_320x240_2cm", "kind": "live", "scene": "room", "w": 320, "h": 240, "mm": 20, "frames": 20},
        # live scanning at full resolution, the whole frame replayed as one graph
        {"name": "graph_640x480_5mm", "kind": "graph", "scene": "desk", "w": 640, "h": 480, "mm": 5, "frames": 16},
        # many robots' rooms served at once, one frame of each per pass
        {"name": "rooms_64_320x240", "kind": "rooms", "n": 64, "w": 320, "h": 240, "frames": 4},
        # live scanning with the probabilistic fusion (outlier model), an odd image size
        {"name": "psdf_333x251_2cm", "kind": "psdf", "scene": "room", "w": 333, "h": 251, "mm": 20, "frames": 20},
        # a new scan: the volume is emptied, the first frames allocate everything they see
        {"name": "scan_640x480_1cm", "kind": "scan", "scene": "desk", "w": 640, "h": 480, "mm": 10, "frames": 4},
        # offline fusion of recorded colour frames, no mesh wanted yet
        {"name": "fuse_640x480_1cm", "kind": "fuse", "scene": "desk", "w": 640, "h": 480, "mm": 10, "frames": 8},
        # denoising a probabilistically fused model before it is exported
        {"name": "denoise_2cm_50", "kind": "denoise", "scene": "room", "w": 320, "h": 240, "mm": 20, "frames": 10,
         "iters": 50},
        # one gradient of the rendered depth against an observation, by pose and by field
        {"name": "adjoint_640x480_1cm", "kind": "adjoint", "scene": "room", "w": 640, "h": 480, "mm": 10, "frames": 10},
        # tracking a new frame against the model from a predicted pose
        {"name": "track_320x240_2cm", "kind": "track", "scene": "room", "w": 320, "h": 240, "mm": 20, "frames": 10,
         "iters": 20},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, most):
    w = _log(rng, 96, most)
    return {"w": w, "h": max(72, int(w * rng.uniform(0.6, 0.9)))}


def draw(rng):
    kind = rng.choice(["render", "live", "graph", "rooms", "psdf", "scan", "fuse", "denoise", "adjoint", "track"])
    if kind == "rooms":
        return {"kind": kind, "n": _log(rng, 2, 40), **_size(rng, 320), "frames": 4}
    c = {"kind": kind, "scene": rng.choice(["room", "desk"]), **_size(rng, 1200 if kind == "render" else 640)}
    if kind in ("psdf", "denoise", "track"):
        c["mm"] = rng.choice([20, 40])
    elif kind in ("live", "adjoint", "scan", "fuse"):
        c["mm"] = rng.choice([10, 20, 40])
    else:
        c["mm"] = rng.choice([5, 10, 20])
    c["frames"] = rng.randint(3, 6) if kind == "scan" else rng.randint(4, 10)
    if kind == "denoise":
        c["iters"] = rng.randint(10, 50)
    if kind == "track":
        c["iters"] = rng.randint(5, 20)
    return c


def _config(case, seed):
    base = C3 if case["kind"] in ("psdf", "denoise") else (C1 if case["scene"] == "room" else C2)
    w, h, mm = case["w"], case["h"], case["mm"]
    buckets, pool, verts = POOLS[mm]
    if base is C3:
        buckets, pool = 4 * buckets, 4 * pool
    elif case["kind"] in ("adjoint", "fuse"):
        pool //= 4 if mm == 10 else 1
    f = 525.0 * w / 640.0
    desk = case["scene"] == "desk"
    return replace(base, width=w, height=h, fx=f, fy=f, cx=0.5 * (w - 1), cy=0.5 * (h - 1), voxel_size=mm / 1000.0,
                   truncation=4 * mm / 1000.0, bucket_count=buckets, value_capacity=pool, max_vertices=verts,
                   max_triangles=2 * verts, frames=300 if desk else 20, synth_kind=1 if desk else 0,
                   hole_fraction=0.02 if desk else base.hole_fraction, seed=1 + seed % 100003)


def _frames(cfg, n, first=0):
    return ([synth_depth(cfg, first + i) for i in range(n)], [synth_pose(cfg, first + i) for i in range(n)])


def _images(cfg, n=1):
    """Depth, vertex and normal images of n raycasts, and their pointers."""
    px = n * cfg.width * cfg.height
    im = {"depth": torch.empty(px, device="cuda"), "vertex": torch.empty(px, 3, device="cuda"),
          "normal": torch.empty(px, 3, device="cuda")}
    return im, [im[k].data_ptr() for k in ("depth", "vertex", "normal")]


def _field(vol, which, typestr="<f4"):
    """A voxel field of the volume as a tensor of one row per pool slot (a view)."""
    ptr, n = vol.field_ptr(which)

    class View:
        __cuda_array_interface__ = {"shape": (n // 512, 512), "typestr": typestr, "data": (ptr, False), "version": 2}

    return torch.as_tensor(View(), device="cuda")


def _rows(case):
    """Rows of a field that is handed out, the same for every scene of a case:
    the blocks of at most ten frames with some room (the rest repeat a row
    that is not in use)."""
    c = (48000 if case["scene"] == "room" else 18000) * 4 if case["kind"] == "denoise" else \
        18000 if case["scene"] == "room" else 3000
    return max(512, c * 100 // case["mm"] ** 2)


def _slots(vol, blocks, rows):
    """Pool slot of each block of dump_blocks (sorted by position): the blocks are
    tagged through load_blocks, read back by slot, and put back as they were."""
    n = len(blocks["pos"])
    if n > rows:
        raise ValueError("%d blocks, more than the %d rows of the case" % (n, rows))
    tag = np.full((n, 512), -1.0, np.float32)
    tag[:, 0] = np.arange(n)
    vol.load_blocks(blocks["pos"], tag, blocks["weight"])
    row = _field(vol, A.MH_FIELD_SDF)
    used = torch.nonzero((row[:, 1] == -1.0) & (row[:, 2] == -1.0)).reshape(-1)
    at = torch.full((rows,), len(row) - 1, dtype=torch.int64, device="cuda")
    at[row[used, 0].long()] = used
    vol.load_blocks(blocks["pos"], blocks["sdf"], blocks["weight"])
    return at


def _fused(cfg, n):
    """A volume with n frames fused, as a scan leaves it."""
    eng = MainEngine(cfg, recycle=False)
    depth, pose = _frames(cfg, n)
    for d, p in zip(depth, pose):
        eng.frame(d, p, mesh=cfg.psdf)
    return eng.vol


def _se3(w, u):
    th = np.linalg.norm(w)
    W = np.array([[0, -w[2], w[1]], [w[2], 0, -w[0]], [-w[1], w[0], 0]])
    T = np.eye(4)
    T[:3, :3] += math.sin(th) / th * W + (1 - math.cos(th)) / th ** 2 * W @ W
    T[:3, 3] = u
    return T


def _moved(pose, rng, degrees, metres):
    """A pose a little off the given one."""
    axis = rng.normal(size=3)
    axis *= np.radians(degrees) / np.linalg.norm(axis)
    u = rng.normal(size=3)
    return (_se3(axis, u * metres / np.linalg.norm(u)) @ pose.astype(np.float64)).astype(np.float32)


def prepare(case, seed):
    kind, n = case["kind"], case["frames"]
    rng = np.random.default_rng(seed)
    s = {"kind": kind, "next": 0, "n": n}
    if kind == "rooms":
        cfgs = [replace(c, width=case["w"], height=case["h"], fx=262.5 * case["w"] / 320.0,
                        fy=262.5 * case["w"] / 320.0, cx=0.5 * case["w"], cy=0.5 * case["h"],
                        seed=1 + (1000 * seed + i) % 1000003)
                for i, c in enumerate(c4_scenes(case["n"], n))]
        depth = np.stack([np.stack([synth_depth(c, f) for c in cfgs]) for f in range(n)])
        s["depth"] = torch.from_numpy(depth.view(np.int16)).cuda()
        s["pose"] = [np.stack([synth_pose(c, f) for c in cfgs]) for f in range(n)]
        s["batch"] = Batch(cfgs)
        s["images"], p = _images(cfgs[0], len(cfgs))
        s["batch"].set_raycast(*p)
        return s
    cfg = _config(case, seed)
    if kind in ("render", "adjoint"):
        s["vol"] = _fused(cfg, n)
        pose = synth_pose(cfg, n // 2)
        s["cTw"] = np.linalg.inv(_moved(pose, rng, 2.0, 0.02).astype(np.float64)).astype(np.float32)
        s["images"], s["ptr"] = _images(cfg)
        if kind == "adjoint":
            s["obs"] = torch.from_numpy(synth_depth(cfg, n // 2) * np.float32(0.001)).cuda()
            s["slots"] = _slots(s["vol"], s["vol"].dump_blocks(), _rows(case))
            s["grad"] = torch.empty(cfg.value_capacity, 512, device="cuda")
        return s
    if kind == "track":
        s["vol"] = _fused(cfg, n)
        s["depth"] = synth_depth(cfg, n // 2)
        s["start"] = _moved(synth_pose(cfg, n // 2), rng, 1.0, 0.02)
        s["iters"] = case["iters"]
        return s
    if kind == "denoise":
        s["vol"] = _fused(cfg, n)
        s["cfg"], s["iters"] = cfg, case["iters"]
        s["blocks"] = s["vol"].dump_blocks()
        s["slots"] = _slots(s["vol"], s["blocks"], _rows(case))
        s["vol"].collect_all()
        return s
    depth, s["pose"] = _frames(cfg, n)
    if kind == "graph":
        s["depth"] = torch.from_numpy(np.stack(depth).view(np.int16)).cuda()
        s["batch"] = Batch([cfg])
        s["images"], p = _images(cfg)
        s["batch"].set_raycast(*p)
        return s
    s["depth"] = depth
    if kind == "fuse":
        s["cfg"], vol = cfg, Volume(cfg)
        s["vol"], s["color"], s["cTw"] = vol, [synth_color(cfg, f) for f in range(n)], []
        for d, p in zip(depth, s["pose"]):  # the blocks of a first pass over the recording
            vol.upload_depth(d, p)
            vol.alloc()
            s["cTw"].append(vol.pose()[1])
        s["blocks"] = vol.dump_blocks()
        s["slots"] = _slots(vol, s["blocks"], _rows(case))
        return s
    s["engine"] = MainEngine(cfg)
    s["images"], s["ptr"] = _images(cfg)
    return s


def run(s):
    kind = s["kind"]
    if kind in ("graph", "rooms"):
        f, b = s["next"], s["batch"]
        s["next"] = (f + 1) % s["n"]
        b.frame(s["depth"][f].data_ptr(), s["pose"][f])
        b.run(mesh=True, raycast=True, graph=True)
        return s["images"]
    if kind in ("live", "psdf"):
        f, e = s["next"], s["engine"]
        s["next"] = (f + 1) % s["n"]
        e.frame(s["depth"][f], s["pose"][f])
        e.vol.raycast(e.vol.pose()[1], *s["ptr"])
        return s["images"]
    if kind == "scan":
        e = s["engine"]
        e.vol.reset()
        e.integrated_frame_count = 0
        for d, p in zip(s["depth"], s["pose"]):
            e.frame(d, p)
        e.vol.raycast(e.vol.pose()[1], *s["ptr"])
        return s["images"]
    vol = s["vol"]
    if kind == "render":
        vol.raycast(s["cTw"], *s["ptr"])
        return s["images"]
    if kind == "adjoint":
        s["grad"].zero_()
        out = vol.raycast_backward(s["cTw"], s["obs"].data_ptr(), s["grad"].data_ptr(), noalloc=True)
        out["grad_sdf"] = s["grad"][s["slots"]]
        return out
    if kind == "track":
        vol.upload_depth(s["depth"], s["start"])
        return vol.localize(s["start"], iterations=s["iters"])
    if kind == "denoise":
        cfg = s["cfg"]
        vol.pd_init()
        for i in range(s["iters"]):
            e = vol.pd_iterate(cfg.pd_lambda, cfg.pd_sigma, cfg.pd_tau, energy=i + 1 == s["iters"])
        return {"sdf": _field(vol, A.MH_FIELD_SDF)[s["slots"]], "energy": np.array(e)}
    for d, c, p in zip(s["depth"], s["color"], s["pose"]):  # fuse
        vol.upload_depth(d, p)
        vol.upload_color(c)
        vol.alloc()
        vol.collect_visible()
        vol.integrate_tsdf()
    return {"sdf": _field(vol, A.MH_FIELD_SDF)[s["slots"]], "weight": _field(vol, A.MH_FIELD_WEIGHT)[s["slots"]],
            "color": _field(vol, A.MH_FIELD_COLOR, "<i4")[s["slots"]]}


def work(case):
    """Bytes and operations from the scene's size: a view sees about 13 m^2 of
    the room or 6 m^2 of the desk, a surface patch of one block's face lies in
    about 2.5 blocks of the truncation band, and about half of their voxels
    are updated by a frame; with outliers a view holds about ten times the
    blocks, most of them in observed free space.  A pixel's march reads its raw depth and writes
    seven values; a meshed block reads its 9^3 corner values and its cube
    words; a rendered block's field is read once."""
    kind = case["kind"]
    px = case["w"] * case["h"]

    def blocks(area, mm):
        return 2.5 * area / (64e-6 * mm * mm)

    def frame(vis, px, mesh=True, view=True):
        b = 24.0 * 256 * vis + 12 * vis + 6 * px
        f = 60.0 * 512 * vis + 100 * px
        if mesh:
            b += 6344.0 * vis
            f += 30.0 * 512 * vis
        if view:
            b += 28.0 * px + 2048.0 * 0.7 * vis
            f += 40.0 * 60 * px
        return b, f

    if kind == "rooms":
        b, f = frame(sum(blocks(13.0, 10 * (1 + k % 4)) for k in range(case["n"])), px * case["n"])
        return {"bytes": b, "flops": f}
    area = 13.0 if case["scene"] == "room" else 6.0
    vis, n = blocks(area, case["mm"]), case["frames"]
    if kind == "render":
        return {"bytes": 28.0 * px + 2048.0 * 0.7 * vis, "flops": 2400.0 * px}
    if kind == "adjoint":
        return {"bytes": 4.0 * px + 4096.0 * 0.7 * vis, "flops": 6000.0 * px}
    if kind == "track":
        return {"bytes": 2.0 * px + 2048.0 * 0.7 * vis, "flops": case["iters"] * 600.0 * px / 4}
    if kind == "denoise":
        seen = vis * (3.3 * n if case["scene"] == "room" else 23)  # blocks of the fused frames
        # per iteration: weight, field, starting field, bar, dual (3) read, dual, bar and field written
        return {"bytes": case["iters"] * seen * 512 * 48.0, "flops": case["iters"] * seen * 512 * 60.0}
    if kind == "fuse":
        b, f = frame(vis, px, False, False)
        return {"bytes": n * (b + 4 * px), "flops": n * f}
    if kind == "scan":
        b, f = frame(vis, px, True, False)
        return {"bytes": n * b + 28 * px, "flops": n * f + 2400 * px}
    if kind == "psdf":
        b, f = frame(10 * vis, px)
        return {"bytes": b, "flops": 2 * f}
    b, f = frame(vis, px)
    return {"bytes": b, "flops": f}


# ------------------------------------------------------------------ 64 bits
# The raycasts have no plain 64-bit counterpart: a pixel is hit or not, and by
# which step, as its 32-bit samples decide.  Fusion and denoising are
# arithmetic on fixed inputs: the choices (pixel, visibility, observed or not)
# follow the 32-bit expressions, the values are 64-bit.
def exact(case, seed):
    if case["kind"] == "fuse":
        return _exact_fuse(prepare(case, seed))
    if case["kind"] == "denoise":
        return _exact_denoise(prepare(case, seed))
    return None


def _pad(s, x):
    """The rows of blocks followed by those of the slot not in use."""
    return torch.cat([x, torch.zeros(len(s["slots"]) - len(x), 512, dtype=x.dtype, device="cuda")])


def _project(cfg, m, x, y, z):
    t = [m[4 * r] * x + m[4 * r + 1] * y + m[4 * r + 2] * z + m[4 * r + 3] for r in range(3)]
    return t[0] * np.float32(cfg.fx) / t[2] + np.float32(cfg.cx), t[1] * np.float32(cfg.fy) / t[2] + np.float32(cfg.cy), t[2]


def _exact_fuse(s):
    cfg = s["cfg"]
    pos = torch.from_numpy(s["blocks"]["pos"]).cuda()
    i = torch.arange(512, device="cuda")
    local = torch.stack([i % 8, i // 8 % 8, i // 64], 1)
    vox = (pos[:, None, :] * 8 + local[None]).int()
    vs = np.float32(cfg.voxel_size)
    x, y, z = [(vox[..., k].float() * float(vs)) for k in range(3)]
    v64 = vox.double() * float(vs)
    sdf = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    wgt = torch.zeros_like(sdf)
    f32 = torch.float32
    tr = float(np.float32(cfg.truncation))
    lo, hi, ub = (float(np.float32(v)) for v in (cfg.min_depth, cfg.max_depth, cfg.sdf_upper_bound))
    half = vs * np.float32(0.5) * np.float32(7.0)
    wm1, hm1 = float(cfg.width - 1), float(cfg.height - 1)
    for d, p, c32 in zip(s["depth"], s["pose"], s["cTw"]):
        m = [torch.tensor(v, dtype=f32, device="cuda") for v in c32.reshape(-1)]
        c64 = np.linalg.inv(p.astype(np.float64))
        corner = [(pos[:, k] * 8).float() * float(vs) + float(half) for k in range(3)]
        bu, bv, bz = _project(cfg, m, *corner)
        nx, ny, nz = (2.0 * bu - wm1) / wm1 * np.float32(0.95), (hm1 - 2.0 * bv) / hm1 * np.float32(0.95), \
            (bz - lo) / float(np.float32(hi) - np.float32(lo)) * np.float32(0.95)
        seen = ((nx.abs() <= 1) & (ny.abs() <= 1) & (nz >= 0) & (nz <= 1))[:, None]
        u, v, zc = _project(cfg, m, x, y, z)
        u, v = torch.trunc(u + 0.5), torch.trunc(v + 0.5)
        inside = (u >= 0) & (u < cfg.width) & (v >= 0) & (v < cfg.height) & seen
        pix = torch.where(inside, v * cfg.width + u, torch.zeros_like(u)).long()
        dm = torch.from_numpy(d.astype(np.float32) * np.float32(0.001)).cuda().reshape(-1)
        dm = torch.where((dm >= lo) & (dm <= hi), dm, torch.full_like(dm, -math.inf))
        dd = dm[pix]
        live = inside & (dd != -math.inf) & (dd != 0) & (dd < ub) & ~(dd - zc <= -tr)
        obs = dd.double() - (c64[2, 0] * v64[..., 0] + c64[2, 1] * v64[..., 1] + c64[2, 2] * v64[..., 2] + c64[2, 3])
        obs = obs.clamp(-tr, tr)
        w = (10.0 * cfg.weight_sample * (1.0 - (dd.double() - lo) / (hi - lo))).clamp(min=1.0)
        new = (sdf * wgt + torch.nan_to_num(obs) * torch.nan_to_num(w)) / (wgt + torch.nan_to_num(w, posinf=1.0))
        sdf = torch.where(live, new, sdf)
        wgt = torch.where(live, wgt + w, wgt)
    return {"sdf": _pad(s, sdf), "weight": _pad(s, wgt), "color": None}


def _exact_denoise(s):
    cfg, b = s["cfg"], s["blocks"]
    pos = b["pos"].astype(np.int64)
    n = len(pos)
    key = lambda q: ((q[:, 0] + 4096) * 8192 + q[:, 1] + 4096) * 8192 + q[:, 2] + 4096  # noqa: E731
    keys = torch.from_numpy(key(pos)).cuda()  # sorted: the blocks are
    i = torch.arange(512, device="cuda")
    local = torch.stack([i % 8, i // 8 % 8, i // 64], 1)

    def neighbour(axis, step):
        q = pos.copy()
        q[:, axis] += step
        want = torch.from_numpy(key(q)).cuda()
        at = torch.searchsorted(keys, want).clamp(max=n - 1)
        at = torch.where(keys[at] == want, at, torch.full_like(at, -1))
        c = local.clone()
        c[:, axis] += step
        out = (c[:, axis] < 0) | (c[:, axis] > 7)
        c[:, axis] %= 8
        li = c[:, 0] + 8 * c[:, 1] + 64 * c[:, 2]
        blk = torch.where(out[None], at[:, None], torch.arange(n, device="cuda")[:, None])
        return torch.where(blk < 0, torch.full_like(blk, -1), blk * 512 + li[None]).reshape(-1)

    fwd = [neighbour(k, +1) for k in range(3)]
    bwd = [neighbour(k, -1) for k in range(3)]
    live = ~(torch.from_numpy(b["weight"].reshape(-1).astype(np.float64)).cuda() < 1e-6)
    sdf = torch.from_numpy(b["sdf"].reshape(-1).astype(np.float64)).cuda()
    s0 = sdf.clone()

    def valid(nb):
        ok = live.clone()
        for j in nb:
            ok &= (j >= 0) & live[j.clamp(min=0)]
        return ok

    okf, okb = valid(fwd), valid(bwd)

    def grad(x):
        return torch.stack([torch.where(okf, x[j.clamp(min=0)] - x, torch.zeros_like(x)) for j in fwd])

    g = grad(sdf)
    w_pd = torch.exp(g.square().sum(0).sqrt() / float(np.float32(cfg.voxel_size)))
    p, bar = torch.zeros_like(g), torch.zeros_like(sdf)
    lam, sigma, tau, alpha = (float(np.float32(v)) for v in (cfg.pd_lambda, cfg.pd_sigma, cfg.pd_tau, 0.02))
    for _ in range(s["iters"]):
        data = torch.where(live, (sdf - s0).square(), torch.zeros_like(sdf)).sum()
        size = grad(sdf).square().sum(0).sqrt()
        tv = torch.where(live, torch.where(size < alpha, 0.5 * size.square() / alpha, size - 0.5 * alpha),
                         torch.zeros_like(sdf)).sum()
        p = (p + sigma * grad(bar)) / (1.0 + sigma * alpha)
        p = p / p.square().sum(0).sqrt().clamp(min=1.0)
        div = sum(p[k][bwd[k].clamp(min=0)] - p[k] for k in range(3))
        div = torch.where(okb, div, torch.zeros_like(div))
        l = lam * w_pd
        new = (sdf - tau * div + l * tau * s0) / (1.0 + l * tau)
        new = torch.where(w_pd > 2.0, s0, new)
        new = torch.where(live, new, sdf)
        bar = torch.where(live, 2.0 * new - sdf, bar)
        sdf = new
    return {"sdf": _pad(s, sdf.reshape(n, 512)), "energy": torch.stack([data, tv, data * lam / 2.0 + tv])}
