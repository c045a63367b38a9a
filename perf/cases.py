"""The work that users of this framework have it do, as cases that can be timed.

A case is a dict of plain values; `prepare` makes what a program has in hand
before the call, `run` is one pass through the public entry points and returns
its outputs whole, `work` says what a pass cannot do without and `exact` gives
the floating outputs in 64 bits.

Kinds of work:
  run     a world is filled by a scene generator and ticked in one captured run
          with periodic state hashes; the grid stays on the device
  upload  a host grid is uploaded, ticked with periodic hashes, and either
          downloaded or handed on by its device pointer
  edit    an interactive program pokes cells and takes single ticks
  play    the viewer loop: some ticks, then a frame, several times
  view    frames of a world that does not move
  sdf     the full-screen sphere tracer
  batch   many independent worlds in one run
  serve   simulation requests submitted to the server, all final hashes
"""
import math

import numpy as np
import torch

import fallingsand3d_amd as F
from fallingsand3d_amd import render as R

DEVICE = "cuda"
# The three palette entries the voxel renderer gives STATIC, SAND and FLUID
# (entries 127, 162 and 137 of the 256-entry table).
COLOURS = {1: (0.52, 0.52, 0.52), 2: (1.0, 0.82, 0.16), 3: (0.0, 0.21, 0.88)}


def listed():
    return [
        # a small world watched tick by tick: 256 ticks, a hash after each
        {"name": "rain64", "kind": "run", "nx": 64, "ny": 64, "nz": 64, "scene": "rain", "dense": False,
         "ticks": 256, "every": 1},
        # an editor on a small odd-sized world: pokes, single ticks, hashes
        {"name": "edit48", "kind": "edit", "nx": 48, "ny": 37, "nz": 29, "rounds": 8},
        # a host program that hands a mid-sized grid over and wants it back
        {"name": "roundtrip192", "kind": "upload", "nx": 192, "ny": 160, "nz": 224, "side": 40, "ticks": 200,
         "every": 50, "back": True},
        # the 512^3 box scene, 1000 ticks, a hash every 50
        {"name": "boxes512", "kind": "upload", "nx": 512, "ny": 512, "nz": 512, "side": 64, "ticks": 1000,
         "every": 50, "back": False},
        # a dense world of odd sizes, every voxel ticked
        {"name": "dense1000", "kind": "run", "nx": 1000, "ny": 701, "nz": 603, "scene": "rain", "dense": True,
         "ticks": 48, "every": 0},
        # the largest single world: collapsing columns at 2048^3
        {"name": "pillars2048", "kind": "run", "nx": 2048, "ny": 2048, "nz": 2048, "scene": "pillars",
         "dense": False, "ticks": 60, "every": 60},
        # a quarter of it with skipping off (a slab of a sharded world)
        {"name": "dense2048", "kind": "run", "nx": 2048, "ny": 2048, "nz": 512, "scene": "pillars", "dense": True,
         "ticks": 32, "every": 0},
        # the viewer loop on a large world: ten ticks, a 1280x720 frame, four times
        {"name": "play1024", "kind": "play", "nx": 1024, "ny": 1024, "nz": 1024, "ticks": 10, "frames": 4,
         "W": 1280, "H": 720},
        # a frame of a landscape that is at rest
        {"name": "view512", "kind": "view", "nx": 512, "ny": 512, "nz": 320, "W": 1280, "H": 720},
        # the sphere tracer at full HD
        {"name": "sdf1080", "kind": "sdf", "W": 1920, "H": 1080},
        # 4096 worlds of uneven sizes, 500 ticks in one autotuned run
        {"name": "batch4096", "kind": "batch", "n": 4096, "lo": 16, "hi": 128, "ticks": 500, "tuned": True},
        # a burst of simulation requests of uneven sizes and lengths
        {"name": "serve1500", "kind": "serve", "n": 1500, "lo": 32, "hi": 256, "tick_lo": 10, "tick_hi": 500},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "upload", "upload", "edit", "play", "view", "sdf", "batch", "batch",
                       "serve"])
    if kind == "run":
        dims = [_log(rng, 24, 2048), _log(rng, 24, 1200), _log(rng, 24, 1200)]
        n = dims[0] * dims[1] * dims[2]
        ticks = max(4, min(300, int(2e10 / n))) + rng.randrange(3)
        return {"kind": kind, "nx": dims[0], "ny": dims[1], "nz": dims[2], "scene": rng.choice(["rain", "pillars"]),
                "dense": rng.random() < 0.4, "ticks": ticks, "every": rng.choice([0, 1, 10, ticks])}
    if kind == "upload":
        dims = [_log(rng, 32, 600) for _ in range(3)]
        ticks = rng.randrange(20, 400)
        return {"kind": kind, "nx": dims[0], "ny": dims[1], "nz": dims[2], "side": max(4, min(dims) // 6),
                "ticks": ticks, "every": rng.choice([0, 7, 50]), "back": rng.random() < 0.5}
    if kind == "edit":
        return {"kind": kind, "nx": _log(rng, 8, 256), "ny": _log(rng, 8, 256), "nz": _log(rng, 8, 256),
                "rounds": rng.randrange(2, 12)}
    if kind == "play":
        return {"kind": kind, "nx": _log(rng, 128, 1024), "ny": _log(rng, 128, 1024), "nz": _log(rng, 128, 1024),
                "ticks": rng.randrange(1, 16), "frames": rng.randrange(2, 5), "W": rng.randrange(320, 1920),
                "H": rng.randrange(200, 1080)}
    if kind == "view":
        return {"kind": kind, "nx": _log(rng, 64, 512), "ny": _log(rng, 64, 512), "nz": _log(rng, 48, 384),
                "W": rng.randrange(320, 1920), "H": rng.randrange(200, 1080)}
    if kind == "sdf":
        return {"kind": kind, "W": rng.randrange(320, 1920), "H": rng.randrange(200, 1080)}
    if kind == "batch":
        lo = _log(rng, 8, 32)
        return {"kind": kind, "n": _log(rng, 24, 4096), "lo": lo, "hi": rng.randrange(lo + 8, 129),
                "ticks": rng.randrange(10, 500), "tuned": rng.random() < 0.3}
    lo = _log(rng, 16, 48)
    return {"kind": "serve", "n": _log(rng, 16, 1500), "lo": lo, "hi": rng.randrange(lo + 16, 257), "tick_lo": 10,
            "tick_hi": rng.randrange(40, 500)}


# ---- inputs -------------------------------------------------------------------------


def _dims(case):
    return case["nx"], case["ny"], case["nz"]


def _pillars(dims, seed):
    """Sand columns over a pool, scaled from the 2048^3 scene's proportions."""
    nx, ny, nz = dims
    m = min(nx, ny)
    r = max(1, m // 64)
    return (max(4, min(256, nx * ny // (64 * r * r))), max(1, r // 8), r, max(2, nz // 8), max(2, nz * 7 // 8),
            max(1, nx // 8), max(1, nx // 3), max(1, ny // 8), max(1, ny // 3), max(1, nz // 64), max(1, nz // 16))


def _fill(w, case, seed):
    if case["scene"] == "rain":
        w.fill_rain(seed, F.threshold(3, 10))
    else:
        w.fill_pillars(seed, _pillars(w.dims, seed))


def _landscape(case, seed):
    """A hilly sand and rock landscape with water in the valleys: g[z][y][x]."""
    nx, ny, nz = _dims(case)
    gen = torch.Generator().manual_seed(int(seed))
    h = torch.zeros(ny, nx)
    for cells, amp in ((4, 0.22), (9, 0.10), (33, 0.03)):
        k = torch.rand(1, 1, cells, cells, generator=gen)
        h += amp * torch.nn.functional.interpolate(k, size=(ny, nx), mode="bicubic", align_corners=True)[0, 0]
    h = (h.clamp(0.02, 0.9) * nz).to(DEVICE)
    z = torch.arange(nz, device=DEVICE, dtype=torch.float32).reshape(nz, 1, 1)
    g = torch.where(z < h - 3, 1, torch.where(z < h, 2, torch.where(z < 0.16 * nz, 3, 0)))
    g[0] = 1
    return g.to(torch.uint8)


def _camera(dims, seed, W, H):
    """An orbit camera as float32 values: origin, basis rows, light, aspect."""
    rng = np.random.default_rng(int(seed) + 77)
    ang, elev = rng.uniform(0, 2 * math.pi), rng.uniform(0.25, 0.6)
    c = np.array(dims, np.float64) * 0.5
    m = float(max(dims))
    eye = c + 1.4 * m * np.array([math.cos(ang) * math.cos(elev), math.sin(ang) * math.cos(elev), math.sin(elev)])
    f = (c - eye) / np.linalg.norm(c - eye)
    left = np.array([-f[1], f[0], 0.0])
    left /= np.linalg.norm(left)
    basis = np.stack([left, np.cross(left, f), f])
    light = c - m * np.array([2.0, 5.0, 3.0])
    return [np.asarray(v, np.float32) for v in (eye, basis, light)] + [float(np.float32(W / H))]


def _sdf_camera(seed):
    rng = np.random.default_rng(int(seed))
    return np.array([rng.uniform(-0.3, 0.3), rng.uniform(-0.3, 0.3), rng.uniform(-3.0, -1.2)], np.float32)


class _Pointer:
    """What a tensor over a world's grid holds on to: the world lives as long as the tensor."""

    def __init__(self, p, w):
        self.w = w
        self.__cuda_array_interface__ = {"shape": w.shape, "typestr": "|u1", "data": (p, False), "strides": None,
                                         "version": 2}


class _DeviceGrid:
    """A world's current grid as a torch tensor over its device pointer."""

    def __init__(self, w):
        self.w, self.seen = w, {}

    def tensor(self):
        p = self.w.device_ptr()
        if p not in self.seen:
            self.seen[p] = torch.as_tensor(_Pointer(p, self.w), device=DEVICE)
        return self.seen[p]


def prepare(case, seed):
    torch.zeros(1, device=DEVICE)
    F.init(0)
    k = case["kind"]
    s = {"case": case, "seed": int(seed)}
    if k in ("run", "upload", "edit", "play", "view"):
        w = F.World(_dims(case), flags=F.DENSE if case.get("dense") else 0)
        s["w"], s["grid"] = w, _DeviceGrid(w)
        if k == "upload":
            w.fill_boxes(s["seed"], side_min=max(2, case["side"] // 8), side_max=case["side"])
            s["host"] = w.download()
        elif k == "edit":
            rng = np.random.default_rng(s["seed"])
            s["pokes"] = [[(int(rng.integers(0, case["nx"])), int(rng.integers(0, case["ny"])),
                            int(rng.integers(1, case["nz"])), int(rng.choice([0, 1, 2, 3]))) for _ in range(3)]
                          for _ in range(case["rounds"])]
        elif k in ("play", "view"):
            cams = [_camera(w.dims, s["seed"] + 1000 * i, case["W"], case["H"])
                    for i in range(case.get("frames", 1))]
            s["cams"] = [R.camera(*c) for c in cams]
            if k == "view":
                w.upload(_landscape(case, s["seed"]).cpu().numpy())
    elif k == "sdf":
        s["cam"] = _sdf_camera(s["seed"])
    elif k == "batch":
        dims, thr, seeds = F.batch_specs(case["n"], s["seed"], case["lo"], case["hi"])
        s["b"], s["thr"], s["seeds"] = F.Batch(dims), thr, seeds
        if case["tuned"]:
            s["b"].fill_rain(seeds, thr)
            s["b"].autotune(trial_ticks=10, cache_file=None)
    else:
        s["specs"] = F.serve_specs(case["n"], s["seed"], case["lo"], case["hi"], case["tick_lo"], case["tick_hi"],
                                   2000.0)
        s["server"] = F.Server(budget_bytes=64 << 30, round_ticks=8, max_active=1 << 14)
    return s


def run(s):
    case = s["case"]
    k = case["kind"]
    if k in ("run", "upload"):
        w = s["w"]
        if k == "run":
            _fill(w, case, s["seed"])
        else:
            w.upload(s["host"])
        w.tick_count = 0
        h = w.run(case["ticks"], case["every"])
        grid = w.download() if case.get("back") else s["grid"].tensor()
        return {"hashes": h.view(np.int64), "grid": grid}
    if k == "edit":
        w = s["w"]
        w.fill_rain(s["seed"], F.threshold(3, 10))
        w.tick_count = 0
        got = []
        for pokes in s["pokes"]:
            for x, y, z, v in pokes:
                w.set_voxel(x, y, z, v)
            w.step(1)
            got.append(w.get_voxel(*pokes[0][:3]))
            got.append(w.tick())
        return {"seen": np.array(got, np.uint64).view(np.int64), "grid": s["grid"].tensor()}
    if k == "play":
        w = s["w"]
        w.fill_pillars(s["seed"], _pillars(w.dims, s["seed"]))
        w.tick_count = 0
        frames = []
        for cam in s["cams"]:
            w.run(case["ticks"], 0)
            rgb, hit, face = R.render(w, cam, case["W"], case["H"])
            frames.append([rgb, hit.view(np.int64), face])
        return {"frames": frames, "grid": s["grid"].tensor()}
    if k == "view":
        rgb, hit, face = R.render(s["w"], s["cams"][0], case["W"], case["H"])
        return {"rgb": rgb, "hit": hit.view(np.int64), "face": face}
    if k == "sdf":
        return R.render_sdf(s["cam"], aspect=case["W"] / case["H"], W=case["W"], H=case["H"])
    if k == "batch":
        b = s["b"]
        b.fill_rain(s["seeds"], s["thr"])
        b.tick_count = 0
        return b.run(case["ticks"]).view(np.int64)
    dims, thr, seeds, ticks, _ = s["specs"]
    srv = s["server"]
    ids = srv.replay(dims, seeds, thr, ticks, np.zeros(len(ticks)))
    res = [srv.result(int(i)) for i in ids]
    return {"status": np.array([r[0] for r in res], np.int32),
            "hashes": np.array([r[1] for r in res], np.uint64).view(np.int64)}


def work(case):
    """Each grid in and out once per call of a pass (fills and uploads write it,
    a run of ticks reads and writes it, a hash or a frame reads it, a download
    reads it); one operation per voxel-update or ray step."""
    k = case["kind"]
    px = case.get("W", 0) * case.get("H", 0)
    if k == "sdf":
        return {"bytes": 16 * px, "flops": 64 * 10 * px}
    if k in ("batch", "serve"):
        rng = np.random.default_rng(1)
        e = np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), (4096, 3)))
        vol = float(e.prod(1).mean()) * case["n"]
        ticks = case["ticks"] if k == "batch" else (case["tick_lo"] + case["tick_hi"]) / 2
        return {"bytes": 3 * vol, "flops": vol * ticks}
    n = case["nx"] * case["ny"] * case["nz"]
    if k == "run" or k == "upload":
        return {"bytes": (4 if case.get("back") else 3) * n, "flops": n * case["ticks"]}
    if k == "edit":
        return {"bytes": n * (1 + 4 * case["rounds"]), "flops": 2 * n * case["rounds"]}
    steps = px * max(_dims(case))
    if k == "view":
        return {"bytes": n + 21 * px, "flops": steps}
    return {"bytes": n * (1 + 3 * case["frames"]) + 21 * px * case["frames"],
            "flops": n * case["ticks"] * case["frames"] + steps * case["frames"]}


# ---- the floating outputs in 64 bits ------------------------------------------------


def _pixel_rays(W, H, aspect):
    u = (W - torch.arange(W, device=DEVICE, dtype=torch.float64) - 0.5) / W * 2 - 1
    v = ((torch.arange(H, device=DEVICE, dtype=torch.float64) + 0.5) / H * 2 - 1) / aspect
    d = torch.stack([u.expand(H, W), v[:, None].expand(H, W), torch.ones(H, W, device=DEVICE, dtype=torch.float64)], -1)
    return d / d.norm(dim=-1, keepdim=True)


def _exact_sdf(case, seed):
    W, H = case["W"], case["H"]
    o = torch.tensor(_sdf_camera(seed), device=DEVICE).double()
    d = _pixel_rays(W, H, float(np.float32(W / H))).reshape(-1, 3)
    t = torch.zeros(len(d), device=DEVICE, dtype=torch.float64)
    live = torch.ones_like(t, dtype=torch.bool)
    rgba = torch.zeros(len(d), 4, device=DEVICE, dtype=torch.float64)
    rgba[:, 3] = 1
    eps = 0.0010000000474974513  # 0.001 as a 32-bit float

    def dist(p):
        return p.norm(dim=-1) - 0.5

    for _ in range(64):
        p = o + t[:, None] * d
        r = dist(p)
        hit = live & (r < eps)
        if hit.any():
            q = p[hit]
            h = torch.eye(3, device=DEVICE, dtype=torch.float64) * eps
            g = torch.stack([dist(q + h[a]) - dist(q - h[a]) for a in range(3)], -1)
            g = g / g.norm(dim=-1, keepdim=True)
            light = q - torch.tensor([2.0, 5.0, 3.0], device=DEVICE, dtype=torch.float64)
            light = light / light.norm(dim=-1, keepdim=True)
            rgba[hit, 0] = (g * light).sum(-1).clamp_min(0.05)
        live = live & ~hit & (t <= 1000)
        t = torch.where(live, t + r, t)
    return rgba.reshape(H, W, 4)


def _exact_view(case, seed):
    """The cell-by-cell ray walk through the landscape, in 64 bits."""
    W, H, dims = case["W"], case["H"], _dims(case)
    g = _landscape(case, seed)
    eye, basis, light, aspect = _camera(dims, seed, W, H)
    dt = dict(device=DEVICE, dtype=torch.float64)
    o, light = torch.tensor(eye, **dt), torch.tensor(light, **dt)
    d = _pixel_rays(W, H, aspect).reshape(-1, 3) @ torch.tensor(basis, **dt)
    d = d / d.norm(dim=-1, keepdim=True)
    n = torch.tensor(dims, device=DEVICE)
    t1, t2 = (0 - o) / d, (n - o) / d
    near, far = torch.minimum(t1, t2), torch.maximum(t1, t2).amin(-1)
    tmin, axis = near.max(-1)
    tmin = tmin.clamp_min(0)
    live = torch.nonzero(tmin <= far).squeeze(-1)
    d, t, axis = d[live], tmin[live], axis[live]
    idx = torch.minimum(torch.floor(o + t[:, None] * d).long().clamp_min(0), n - 1)
    step = torch.sign(d).long()
    tnext = (idx + (step > 0) - o) / d
    tdelta = (1 / d).abs()
    colour = torch.zeros(4, 3, **dt)
    for m, c in COLOURS.items():
        colour[m] = torch.tensor(c, **dt)
    out = torch.zeros(H * W, 3, **dt)
    while len(live):
        m = g[idx[:, 2], idx[:, 1], idx[:, 0]].long()
        hit = m > 0
        if hit.any():
            dh, a = d[hit], axis[hit]
            q = o + t[hit][:, None] * dh
            nrm = torch.zeros_like(dh).scatter_(1, a[:, None], -torch.sign(dh.gather(1, a[:, None])))
            ld = q - light
            ld = ld / ld.norm(dim=-1, keepdim=True)
            out[live[hit]] = colour[m[hit]] * (nrm * ld).sum(-1).clamp_min(0.05)[:, None]
        axis = tnext.argmin(-1)
        t = tnext.gather(1, axis[:, None]).squeeze(1)
        idx = idx.scatter_add(1, axis[:, None], step.gather(1, axis[:, None]))
        tnext = tnext.scatter_add(1, axis[:, None], tdelta.gather(1, axis[:, None]))
        keep = ~hit & ((idx >= 0) & (idx < n)).all(-1)
        live, d, t, axis, idx, step, tnext, tdelta = (v[keep] for v in (live, d, t, axis, idx, step, tnext, tdelta))
    return out.reshape(H, W, 3)


def exact(case, seed):
    if case["kind"] == "sdf":
        return _exact_sdf(case, seed)
    if case["kind"] == "view":
        return {"rgb": _exact_view(case, seed), "hit": None, "face": None}
    return None  # whole numbers, or frames after ticks that take too long to follow outside the library
