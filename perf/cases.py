"""Performance cases of the Gaussian point splatting renderer.

Each case is work that a program using this package has it do, through the
package's public entry points: single frames (`Pass.render` and a resolve), a
fly-through with occlusion culling and TAA, whole-scene render requests, a
batch of views, the render server, the allocation-free frame, the two resolves
alone and the load-time BVH order.  Scenes follow the distributions of
`gps_amd.workloads` (uniform box, clustered cube), in Morton load order except
where the order itself is computed.

A program opens a scene once and renders it from many cameras, so the resident
scene belongs to the case (generated on the GPU from the case's sizes, kept
for the next state of the same case); the pass, the cameras, the RNG frame
numbers and the output buffers belong to the state and come from the seed.
"""
import ctypes
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "gaussian-point-splatting_amd"))
import gps_amd as G  # noqa: E402

FORMATS = {"fp32": G.FORMAT_FP32, "half_fp8": G.FORMAT_HALF_FP8, "quantized": G.FORMAT_QUANTIZED}
# resident bytes of one Gaussian: geometry and SH as the formats store them
GEOMETRY_BYTES = {"fp32": 44, "half_fp8": 28, "quantized": 17}


# ----------------------------------------------------------------- cases
def _frame(name, n, scene, fmt, sh, w, h, ss, spp, **kw):
    c = {"name": name, "kind": "frame", "n": n, "scene": scene, "fmt": fmt, "sh": sh, "w": w, "h": h, "ss": ss,
         "spp": spp, "hier": False, "unbiased": True, "reduce": True, "cull_small": False}
    c.update(kw)
    return c


def listed():
    return [
        # The smallest frame a program asks for (thumbnail, first smoke test): launches and latency.
        _frame("thumbnail_20k", 20_000, "uniform", "fp32", 0, 320, 180, 1, 1),
        # A frame inside code that may not allocate (graph capture, serving loop), odd size.
        {"name": "noalloc_301k", "kind": "noalloc", "n": 301_001, "scene": "uniform", "fmt": "half_fp8", "sh": 1,
         "w": 1279, "h": 719, "ss": 1, "spp": 1},
        # The viewer's plain frame: 1M SH0 Gaussians at 720p, one sample per pixel.
        _frame("frame_1m_720p", 1_000_000, "uniform", "fp32", 0, 1280, 720, 1, 1),
        # The quality frame: 10M SH3 Gaussians in fp32 at 1080p, supersampled, 4 samples per pixel.
        _frame("frame_10m_sh3_4spp", 10_000_000, "clustered", "fp32", 3, 1920, 1080, 2, 4),
        # The reference's compressed scene (its default build) at a ragged size, small-Gaussian culling on.
        _frame("quantized_3m_ragged", 3_000_017, "clustered", "quantized", 3, 1501, 843, 2, 2, cull_small=True,
               hier=True),
        # The biased splat (use_unbiased_2d_splatting off), which adds colours per sample.
        _frame("biased_2m", 2_000_003, "clustered", "fp32", 1, 1280, 720, 2, 1, unbiased=False),
        # A served whole-scene request, 4 samples per pixel: many points per framebuffer word.
        _frame("request_25m_4spp", 25_000_000, "clustered", "half_fp8", 3, 1280, 720, 2, 4, hier=True),
        # Real-time camera path: occlusion culling, block culling, TAA, one frame per pass.
        {"name": "flythrough_25m", "kind": "fly", "n": 25_000_000, "scene": "clustered", "fmt": "half_fp8", "sh": 3,
         "w": 1920, "h": 1080, "ss": 2, "spp": 1, "gpb": 1024},
        # Many views of one scene per call (training-set renders, light probes): mixed sizes and spp.
        {"name": "batch_16_views", "kind": "batch", "n": 5_000_000, "scene": "clustered", "fmt": "half_fp8", "sh": 3,
         "views": 16, "ss": 2},
        # Requests against two resident scenes through the serving loop, images back in host memory.
        {"name": "serve_12_requests", "kind": "serve", "n": 1_000_000, "n2": 4_000_000, "requests": 12, "slots": 4},
        # Load time: the reference's default order of a scene, from and to host arrays.
        {"name": "load_order_4m", "kind": "order", "n": 4_000_000, "scene": "clustered"},
        # The resolves alone, 4K output: TAA, then a progressive accumulation step.
        {"name": "resolve_4k", "kind": "resolve", "w": 3840, "h": 2160},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "frame", "noalloc", "fly", "batch", "serve", "order", "resolve"])
    scene = rng.choice(["uniform", "clustered"])
    fmt = rng.choice(["fp32", "half_fp8", "quantized"])
    sh = rng.randrange(4)
    if kind == "frame":
        n = _log(rng, 20_000, 25_000_000 if fmt == "half_fp8" else 8_000_000)
        w, ss, spp = _log(rng, 320, 1920), rng.choice([1, 1, 2, 2, 3]), rng.choice([1, 1, 2, 3, 4])
        if ss == 3:
            w = min(w, 1280)
        return {"kind": kind, "n": n, "scene": scene, "fmt": fmt, "sh": sh, "w": w,
                "h": max(180, int(w * rng.uniform(0.45, 0.75))), "ss": ss, "spp": spp, "hier": rng.random() < 0.5,
                "unbiased": rng.random() < 0.85, "reduce": n > 1_000_000 or rng.random() < 0.8, "cull_small": rng.random() < 0.3}
    if kind == "noalloc":
        w = _log(rng, 320, 1920)
        return {"kind": kind, "n": _log(rng, 10_000, 500_000), "scene": scene, "fmt": fmt, "sh": sh, "w": w,
                "h": max(180, int(w * rng.uniform(0.4, 0.56))), "ss": 1, "spp": 1}
    if kind == "fly":
        w = _log(rng, 640, 1920)
        return {"kind": kind, "n": _log(rng, 500_000, 25_000_000), "scene": "clustered", "fmt": "half_fp8", "sh": sh,
                "w": w, "h": int(w * rng.uniform(0.5, 0.75)), "ss": rng.choice([1, 2]), "spp": rng.choice([1, 1, 2]),
                "gpb": rng.choice([0, 256, 1000, 1024])}
    if kind == "batch":
        return {"kind": kind, "n": _log(rng, 100_000, 5_000_000), "scene": "clustered", "fmt": fmt, "sh": sh,
                "views": _log(rng, 2, 16), "ss": rng.choice([1, 2])}
    if kind == "serve":
        return {"kind": kind, "n": _log(rng, 100_000, 1_000_000), "n2": _log(rng, 1_000_000, 4_000_000),
                "requests": _log(rng, 4, 16), "slots": rng.choice([1, 2, 4])}
    if kind == "order":
        return {"kind": kind, "n": _log(rng, 30_000, 6_000_000), "scene": scene}
    w = _log(rng, 320, 3840)
    return {"kind": "resolve", "w": w, "h": max(180, int(w * rng.uniform(0.4, 0.75)))}


# ----------------------------------------------------------------- scenes
def _spread21(v):
    for s, m in ((32, 0x1F00000000FFFF), (16, 0x1F0000FF0000FF), (8, 0x100F00F00F00F00F), (4, 0x10C30C30C30C30C3),
                 (2, 0x1249249249249249)):
        v = (v | (v << s)) & m
    return v


def _host_arrays(n, scene, sh, morton=True, seed=1):
    """A synthetic scene as host arrays (gps_amd.workloads' distributions)."""
    g = torch.Generator(device="cuda").manual_seed(7919 * seed + n)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=g)

    def uniform(*shape):
        return torch.rand(*shape, device="cuda", generator=g)

    if scene == "uniform":
        means, mu, sigma, op_sigma = (2 * uniform(n, 3) - 1) * 10.0, -4.0, 0.5, 1.0
    else:
        centres = (2 * uniform(max(1, n // 5000), 3) - 1) * 100.0
        which = torch.randint(centres.shape[0], (n,), device="cuda", generator=g)
        means, mu, sigma, op_sigma = centres[which] + 2.0 * normal(n, 3), -3.0, 0.7, 1.5
        del which
    if morton:
        lo, hi = means.amin(0), means.amax(0)
        q = ((means - lo) / (hi - lo) * 2097151.0).to(torch.int64).clamp_(0, 2097151)
        code = _spread21(q[:, 0]) | (_spread21(q[:, 1]) << 1) | (_spread21(q[:, 2]) << 2)
        means = means[torch.argsort(code)]
        del q, code
    rot = normal(n, 4)
    rot /= rot.norm(dim=1, keepdim=True)
    scales = torch.exp(mu + sigma * normal(n, 3))
    ops = torch.sigmoid(op_sigma * normal(n))
    nc = (sh + 1) ** 2
    shs = 0.05 * normal(n, 3 * nc)
    shs[:, :3] *= 6.0
    return G.SceneArrays(*[t.contiguous().cpu().numpy() for t in (means, rot, scales, ops, shs)], sh)


_resident = {}  # the open scenes (and server) of the case at hand


def _open(key, make):
    if key not in _resident:
        if len(_resident) >= 2:
            _resident.clear()
        _resident[key] = make()
    return _resident[key]


def _scene(n, scene, fmt, sh):
    def make():
        chunk = 1 << 23
        if n <= chunk:
            return G.Scene(_host_arrays(n, scene, sh), FORMATS[fmt])
        a = _host_arrays(n, scene, sh)
        s = G.Scene.empty(n, sh, FORMATS[fmt])
        if fmt == "quantized":
            s.set_quantized_bounds(G.quantized_bounds(a))
        for b in range(0, n, chunk):
            s.upload_range(b, a.subset(slice(b, min(n, b + chunk))))
        return s
    return _open((n, scene, fmt, sh), make)


class _Buffer:
    """A torch tensor where the package takes a device array."""

    def __init__(self, shape, dtype=torch.float32):
        self.tensor = torch.zeros(shape, dtype=dtype, device="cuda")
        self.ptr = ctypes.c_void_p(self.tensor.data_ptr())


def _images(w, h):
    return _Buffer((h, w, 3)), _Buffer((h, w)), _Buffer((h, w, 3), torch.uint8)


def _stream():
    if not hasattr(_stream, "it"):
        _stream.it = G.Stream()  # the program's render stream
    return _stream.it


def _eye(r, scene):
    """A camera on the sphere around the scene that it is viewed from."""
    d = [r.gauss(0, 1) for _ in range(3)]
    k = (30.0 if scene == "uniform" else 350.0) / math.sqrt(sum(v * v for v in d))
    return tuple(k * v for v in d)


# ----------------------------------------------------------------- states
def prepare(case, seed):
    r = random.Random(seed * 1000003 + 17)
    s = {"kind": case["kind"]}
    kind = case["kind"]
    if kind in ("frame", "noalloc"):
        w, h, ss, spp = case["w"], case["h"], case["ss"], case["spp"]
        s["scene"] = _scene(case["n"], case["scene"], case["fmt"], case["sh"])
        s["frame"] = G.frame_params(_eye(r, case["scene"]), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 45.0, w, h, ss=ss,
                                    frame=r.randrange(1, 1000), hierarchical=case.get("hier", False),
                                    unbiased=case.get("unbiased", True), reduce_point_count=case.get("reduce", True),
                                    cull_small=case.get("cull_small", False), background=(0.1, 0.2, 0.3), spp=spp)
        s["out"] = _images(w, h)
        s["accum"] = _Buffer((h, w, 3))
        if kind == "frame":
            s["pass"] = G.Pass(G.RenderSettings(w, h, spp, ss,
                                                fully_disable_hierarchical_culling=not case["hier"]), s["scene"])
    elif kind == "fly":
        w, h = case["w"], case["h"]
        s["scene"] = _scene(case["n"], case["scene"], case["fmt"], case["sh"])
        x, y, z = -280.0 + r.uniform(0, 40), r.uniform(-20, 20), r.uniform(-20, 20)
        path = [(x + 4.5 * i, y, z) for i in range(8)]
        path = path + path[-2:0:-1]  # there and back
        s["frames"] = [G.frame_params(e, (e[0] + 1.0, e[1], e[2]), (0.0, 1.0, 0.0), 45.0, w, h, ss=case["ss"],
                                      occlusion=True, hierarchical=True) for e in path]
        s["pass"] = G.Pass(G.RenderSettings(w, h, case["spp"], case["ss"], gaussians_per_block=case["gpb"]),
                           s["scene"])
        s["color"], s["hist"] = ([_Buffer((h, w, 3)) for _ in range(2)] for _ in range(2))
        s["depth"] = [_Buffer((h, w)) for _ in range(2)]
        s["rgb"] = _Buffer((h, w, 3), torch.uint8)
        s["prev_vp"], s["done"], s["size"] = np.zeros(16, np.float32), 0, (w, h)
    elif kind == "batch":
        s["scene"] = _scene(case["n"], case["scene"], case["fmt"], case["sh"])
        lay = random.Random(case["views"])  # the views' sizes belong to the program, the cameras to the seed
        s["frames"], s["out"] = [], []
        for v in range(case["views"]):
            w, h = lay.choice([(854, 480), (1280, 720), (1920, 1080), (641, 479)])
            e = _eye(r, case["scene"])
            s["frames"].append(G.frame_params(tuple(0.43 * c for c in e), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 45.0, w,
                                              h, ss=case["ss"], frame=r.randrange(1, 1000), hierarchical=True,
                                              spp=lay.choice([1, 2, 4])))
            s["out"].append((_Buffer((h, w, 3)), _Buffer((h, w))))
        s["batch"] = G.Batch(s["scene"], case["views"], 1920, 1080, 4, case["ss"])
        s["batch"].set_tuning(256, 4, True)
    elif kind == "serve":
        def make():
            a = G.Scene(_host_arrays(case["n"], "uniform", 0), G.FORMAT_FP32)
            b = G.Scene(_host_arrays(case["n2"], "clustered", 3), G.FORMAT_HALF_FP8)
            server = G.Server(slots=case["slots"], hbm_budget_bytes=24 << 30)
            ids = [server.add_scene(a), server.add_scene(b)]
            server.prepare()
            server.start()
            return server, ids
        s["server"], ids = _open(("serve", case["n"], case["n2"], case["slots"]), make)
        s["requests"] = []
        lay = random.Random(case["requests"])
        for _ in range(case["requests"]):
            k = lay.randrange(2)
            w, h = lay.choice([(854, 480), (1280, 720), (1920, 1080)])
            f = G.frame_params(_eye(r, ("uniform", "clustered")[k]), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 45.0, w, h,
                               ss=2, frame=r.randrange(1, 1000), hierarchical=True, spp=lay.choice([1, 4]))
            s["requests"].append((ids[k], f, np.zeros((h, w, 3), np.uint8)))
    elif kind == "order":
        s["arrays"] = _host_arrays(case["n"], case["scene"], 0, morton=False, seed=seed)
    else:
        w, h = case["w"], case["h"]
        g = torch.Generator(device="cuda").manual_seed(seed)

        def image(*shape):
            b = _Buffer(shape)
            b.tensor.copy_(torch.rand(shape, device="cuda", generator=g))
            return b
        s["size"] = (w, h)
        s["cur"], s["prev"], s["sum"] = image(h, w, 3), image(h, w, 3), image(h, w, 3)
        s["depth"], s["prev_depth"] = _Buffer((h, w)), _Buffer((h, w))
        # NDC depths of surfaces between 5 and 400 units away, in patches
        z = 5.0 + 395.0 * torch.rand((h // 16 + 1, w // 16 + 1), device="cuda", generator=g)
        z = z.repeat_interleave(16, 0).repeat_interleave(16, 1)[:h, :w]
        far, near = 1e4, 0.2
        s["depth"].tensor.copy_((far + near) / (far - near) - 2 * far * near / ((far - near) * z))
        s["out"], s["rgb"], s["rgb2"] = _Buffer((h, w, 3)), _Buffer((h, w, 3), torch.uint8), \
            _Buffer((h, w, 3), torch.uint8)
        x, y = r.uniform(-1, 1), r.uniform(-1, 1)
        a, b = (G.frame_params((x + d, y, -300.0), (0.0, 0.0, 0.0), (0.0, 1.0, 0.0), 45.0, w, h) for d in (0.0, 0.7))
        s["proj"], s["view"] = np.array(b.proj, np.float32), np.array(b.view, np.float32)
        s["prev_vp"] = G.mat4_mul(np.array(a.proj, np.float32), np.array(a.view, np.float32))
    return s


def run(s):
    kind = s["kind"]
    st = _stream()
    if kind == "frame":
        color, depth, rgb = s["out"]
        f = s["frame"]
        f.frame += 1
        s["pass"].render(f, color, depth, st)
        G.resolve_progressive(color, s["accum"], f.width, f.height, 1, rgb, st)
        return {"color": color.tensor, "depth": depth.tensor, "rgb": rgb.tensor}
    if kind == "noalloc":
        color, depth, rgb = s["out"]
        f = s["frame"]
        f.frame += 1
        G.check(G.lib.gps_frame_render_noalloc(s["scene"].handle, ctypes.byref(f), ctypes.c_int64(1 << 24),
                                               color.ptr, depth.ptr, st.handle), "frame")
        return {"color": color.tensor, "depth": depth.tensor}
    if kind == "fly":
        w, h = s["size"]
        f = s["frames"][s["done"] % len(s["frames"])]
        s["done"] += 1
        f.frame = s["done"]
        a = s["done"] % 2
        b = 1 - a
        s["pass"].render(f, s["color"][a], s["depth"][b], st)
        view, proj = np.array(f.view, np.float32), np.array(f.proj, np.float32)
        G.resolve_taa(s["color"][a], s["depth"][a], s["hist"][b], s["depth"][b],
                      G.taa_reprojection(s["prev_vp"], view, proj), 0.9, w, h, s["done"], s["hist"][a], s["rgb"], st)
        s["prev_vp"] = G.mat4_mul(proj, view)
        return {"color": s["color"][a].tensor, "depth": s["depth"][b].tensor, "history": s["hist"][a].tensor,
                "rgb": s["rgb"].tensor}
    if kind == "batch":
        for f in s["frames"]:
            f.frame += 1
        s["batch"].render(s["frames"], [c for c, _ in s["out"]], [d for _, d in s["out"]], st)
        return [(c.tensor, d.tensor) for c, d in s["out"]]
    if kind == "serve":
        server = s["server"]
        for scene, f, image in s["requests"]:
            server.submit(scene, f, out_rgb8=image)
        left = len(s["requests"])
        while left:
            done = server.poll(wait_ms=1000)
            for d in done:
                G.check(d["status"], "request")
            left -= len(done)
        return [image for _, _, image in s["requests"]]
    if kind == "order":
        return s["arrays"].bvh_order().view(np.int32)
    w, h = s["size"]
    G.resolve_taa(s["cur"], s["depth"], s["prev"], s["prev_depth"],
                  G.taa_reprojection(s["prev_vp"], s["view"], s["proj"]), 0.9, w, h, 2, s["out"], s["rgb"], st)
    G.resolve_progressive(s["out"], s["sum"], w, h, 4, s["rgb2"], st)
    return {"out": s["out"].tensor, "rgb": s["rgb"].tensor, "rgb2": s["rgb2"].tensor}


# ----------------------------------------------------------------- work
def _scene_bytes(n, fmt, sh):
    nc = 3 * (sh + 1) ** 2
    colour = {"fp32": 4 * nc, "half_fp8": 10 + nc - 3, "quantized": 57}[fmt]
    return n * (GEOMETRY_BYTES[fmt] + colour)


def work(case):
    """Inputs read once, outputs written once; a projection is about 250
    operations, and a Gaussian of these scenes splats a few samples of about
    100 operations per view."""
    kind = case["kind"]
    if kind in ("frame", "noalloc", "fly"):
        px = case["w"] * case["h"]
        samples = case["ss"] ** 2 * case["spp"]
        return {"bytes": _scene_bytes(case["n"], case["fmt"], case["sh"]) + 19 * px + (12 * px if kind == "fly" else 0),
                "flops": case["n"] * 250.0 + 100.0 * samples * min(case["n"], 4 * px)}
    if kind == "batch":
        px = case["views"] * 1_000_000
        return {"bytes": _scene_bytes(case["n"], case["fmt"], case["sh"]) + 16 * px,
                "flops": case["views"] * case["n"] * 250.0 + 1000.0 * px}
    if kind == "serve":
        n = case["requests"] * (case["n"] + case["n2"]) / 2
        px = case["requests"] * 1_000_000
        return {"bytes": n * 60 + 3 * px, "flops": n * 250.0 + 1000.0 * px}
    if kind == "order":
        return {"bytes": 44 * case["n"], "flops": case["n"] * 100.0 * max(1.0, math.log2(case["n"] / 4))}
    px = case["w"] * case["h"]
    return {"bytes": px * (12 + 4 + 12 + 12 + 12 + 6), "flops": px * 150.0}


# ----------------------------------------------------------------- exact
def exact(case, seed):
    """The resolves in 64 bits.  A rendered image has no such value (its
    samples are 32-bit random streams put into pixels by comparisons), nor
    has an order."""
    if case["kind"] != "resolve":
        return None
    s = prepare(case, seed)
    w, h = s["size"]
    d = torch.float64
    cur, prev, depth = s["cur"].tensor.to(d), s["prev"].tensor.to(d), s["depth"].tensor.to(d)
    M = torch.from_numpy(G.taa_reprojection(s["prev_vp"], s["view"], s["proj"])).to(d).view(4, 4)  # columns
    x = torch.arange(w, device="cuda", dtype=d)[None, :].expand(h, w)
    y = torch.arange(h, device="cuda", dtype=d)[:, None].expand(h, w)
    cx, cy = (x + 0.5) / w * 2 - 1, (y + 0.5) / h * 2 - 1
    p = [M[0, i] * cx + M[1, i] * cy + M[2, i] * depth + M[3, i] for i in (0, 1, 3)]
    px, py = (p[0] / p[2] * 0.5 + 0.5) * w - 0.5, (p[1] / p[2] * 0.5 + 0.5) * h - 0.5
    inside = (px >= 0) & (px < w) & (py >= 0) & (py < h)
    fx, fy = px.floor(), py.floor()
    tx, ty = (px - fx)[..., None], (py - fy)[..., None]
    x0, y0 = fx.long().clamp(0, w - 1), fy.long().clamp(0, h - 1)
    x1, y1 = (fx.long() + 1).clamp(0, w - 1), (fy.long() + 1).clamp(0, h - 1)
    hist = (prev[y0, x0] * (1 - tx) + prev[y0, x1] * tx) * (1 - ty) + (prev[y1, x0] * (1 - tx) + prev[y1, x1] * tx) * ty
    c = cur.permute(2, 0, 1)[None]
    hi = torch.nn.functional.max_pool2d(c, 3, 1, 1)[0].permute(1, 2, 0)
    lo = -torch.nn.functional.max_pool2d(-c, 3, 1, 1)[0].permute(1, 2, 0)
    hist = torch.minimum(torch.maximum(hist, lo - 0.05), hi + 0.05)
    out = torch.where(inside[..., None], cur * 0.1 + hist * 0.9, cur)
    return {"out": out + s["sum"].tensor.to(d), "rgb": None, "rgb2": None}
