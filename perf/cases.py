"""The work a user of this framework has it do, as cases that can be timed and compared.

Frames of one mesh from the smallest the tests draw (a 960-face sphere at 512x512) to the
largest the benchmark does (4M triangles at 4096x4096): one eager call, a captured run of
frames, the spin loop, draw_frame's own host-buffer form, a second mesh drawn onto the
first one's buffers; batches of many meshes, eager and captured; normal-mapped frames with
64 lights shaded by the light loop and by the learned network; and that network's training.

listed() are the cases, draw(rng) gives one more from the same ranges, prepare(case, seed)
makes what a program has in hand before the call, run(state) is one pass through the public
entry points, work(case) what a pass cannot do without, exact(case, seed) its depths (or
training results) in 64-bit arithmetic.
"""
import math

import numpy as np
import torch

import rasteriser_amd as rz
from rasteriser_amd import scenes

MLP_LAYERS = ((64, 12), (64,), (64, 64), (64,), (3, 64), (3,))   # W1 b1 W2 b2 W3 b3
MLP_FLOPS = 2 * (12 * 64 + 64 * 64 + 64 * 3)


def listed():
    def frame(name, **kw):
        c = {"name": name, "kind": "frame", "mesh": "icosphere", "detail": 6, "width": 1920, "height": 1080, "lights": 3,
             "texture": 1024, "normal_map": False, "flat": False, "call": "device", "mlp": False}
        c.update(kw)
        return c

    return [
        # the smallest call: a small preview frame, each waited for
        frame("sphere_512", mesh="uv_sphere", detail=0, width=512, height=512, texture=0),
        # an interactive viewer: one frame of the spin loop per pass, the rotation advancing
        frame("spin_1080p", call="spin"),
        # the benchmark's headline: a turntable of 1080p frames captured as one graph
        frame("turntable_1080p", call="graph", frames=20),
        # draw_frame as the reference calls it: frame and depth in host memory
        frame("host_1080p", call="host"),
        # a scene of two meshes, the second drawn onto the first one's frame and depth: odd
        # size, flat normals, face ids
        frame("overlay_1283x719", detail=5, width=1283, height=719, flat=True, texture=300, call="overlay", lights=5),
        # few, large, thin and partly off-screen triangles: close-ups, ground planes
        frame("large_triangles_1024", mesh="large", detail=3000, width=1024, height=1024, lights=1, texture=0),
        # the largest frame, queued without waiting: scanned or simulated geometry, triangles of about a pixel
        frame("pixels_4m_4096", mesh="soup", detail=4_000_000, width=4096, height=4096, lights=1, texture=0, call="async"),
        # a detailed shot: normal map and 64 lights, by the light loop and by the network
        frame("normal_map_64_lights", lights=64, normal_map=True, call="async"),
        frame("learned_64_lights", lights=64, normal_map=True, call="async", mlp=True),
        # many views or assets at once: a rendering service's batch, tuned and captured once,
        # and a small one whose meshes change from call to call
        {"name": "batch_128_graph", "kind": "batch", "meshes": 128, "max_faces": 200_000, "call": "graph", "ids": False},
        {"name": "batch_12_eager", "kind": "batch", "meshes": 12, "max_faces": 50_000, "call": "eager", "ids": True},
        # fitting the network to a scene: a burst of training steps from given weights
        {"name": "train_8x16384", "kind": "train", "samples": 1 << 18, "batch": 16384, "steps": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame"] * 6 + ["batch"] * 2 + ["train"])
    if kind == "train":
        return {"kind": "train", "samples": _log_int(rng, 5000, 1 << 18), "batch": 64 * _log_int(rng, 1, 255), "steps": rng.randint(1, 8)}
    if kind == "batch":
        return {"kind": "batch", "meshes": _log_int(rng, 2, 100), "max_faces": _log_int(rng, 2000, 200_000),
                "call": rng.choice(["graph", "eager"]), "ids": rng.random() < 0.5}
    c = {"kind": "frame", "mesh": rng.choice(["uv_sphere", "icosphere", "icosphere", "icosphere", "large", "soup"]),
         "width": _log_int(rng, 200, 2600), "height": _log_int(rng, 200, 1500), "lights": _log_int(rng, 1, 80),
         "texture": 0, "normal_map": False, "flat": False, "mlp": False, "call": rng.choice(["device", "async", "spin", "graph", "host", "overlay"])}
    if c["mesh"] == "uv_sphere":
        c.update(detail=0, flat=rng.random() < 0.3)
    elif c["mesh"] == "icosphere":
        c.update(detail=rng.randint(2, 7), texture=rng.choice([0, 64, 333, 1024]), flat=rng.random() < 0.3)
        c["normal_map"] = c["texture"] > 0 and rng.random() < 0.4
        c["mlp"] = c["call"] in ("device", "async", "graph") and rng.random() < 0.25
    else:   # screen-space meshes: square images
        c["width"] = c["height"] = _log_int(rng, 256, 2048)
        c["detail"] = _log_int(rng, 200, 4000) if c["mesh"] == "large" else _log_int(rng, 2000, 1_000_000)
    if c["call"] == "graph":
        c["frames"] = rng.randint(1, 8)
    return c


# ---- inputs -------------------------------------------------------------------------


def _scene(case, seed):
    """(Scene, Args) of a frame case, a function of the seed alone."""
    W, H, flat = case["width"], case["height"], case["flat"]
    if case["mesh"] == "uv_sphere":
        scene, args = scenes.uv_sphere_scene(seed, W, H)
        rng = scenes.SplitMix64(seed)
        scene.lights = scenes.random_lights(rng, case["lights"])
        args = rz.make_args(W, H, fovy=60.0, z_near=0.1, z_far=100.0, flat=flat, angles=scenes.random_angles(rng))
    elif case["mesh"] == "icosphere":
        tex = case["texture"]
        make = scenes.learned_shading_scene if case["normal_map"] else scenes.icosphere_scene
        size = {"map_size": tex} if case["normal_map"] else {"texture_size": max(tex, 2)}
        scene, args = make(seed=seed, width=W, height=H, subdivisions=case["detail"], lights=case["lights"], **size)
        args.flat = int(flat)
        if not tex:
            scene.materials[0].texture = None
    elif case["mesh"] == "large":
        scene, args = scenes.large_triangle_scene(seed, case["detail"], W)
    else:
        scene, args = scenes.screen_soup_scene(seed, case["detail"], W)
    if scene.raster_space and case["lights"] > 1:
        scene.lights = scenes.random_lights(scenes.SplitMix64(seed), case["lights"])
    return scene, args


def _second(case, seed):
    """The mesh drawn second in an overlay: another one of the same kind, over the same image."""
    return _scene(dict(case), seed + 7919)


def _weights(seed):
    """He-uniform weights, small biases, mid-grey output (the network before and during fitting)."""
    rng = np.random.default_rng(seed)
    parts = [rng.uniform(-1, 1, s) * (math.sqrt(6 / s[1]) if len(s) > 1 else 0.1) for s in MLP_LAYERS]
    parts[4] *= 0.3
    parts[5] += 0.4
    return np.concatenate([p.ravel() for p in parts]).astype(np.float32)


def _samples(n, seed):
    """n shaded fragments (n, 15): unit normal, view vector, albedo, normal-map sample, and the
    colour eight lights give them, as bytes / 255."""
    rng = np.random.default_rng(seed)

    def unit(v):
        return v / np.linalg.norm(v, axis=1, keepdims=True)

    nrm = unit(rng.normal(size=(n, 3)))
    nrm[:, 2] = np.abs(nrm[:, 2])
    view = unit(rng.normal(size=(n, 3)) * [0.2, 0.2, 0.05] + [0.0, 0.0, 1.0])
    alb = rng.uniform(0, 1, (n, 3))
    cz = rng.uniform(math.cos(math.radians(30.0)), 1.0, n)
    phi = rng.uniform(0, 2 * math.pi, n)
    sz = np.sqrt(1 - cz * cz)
    bump = np.stack([sz * np.cos(phi), sz * np.sin(phi), cz], 1)
    dirs = unit(rng.normal(size=(8, 3)))
    cols = rng.uniform(0, 1, (8, 3)) * rng.uniform(0.2, 1, (8, 1))
    col = np.floor(np.clip(alb * (np.maximum(nrm @ dirs.T, 0) @ cols), 0, 1) * 255) / 255
    return np.concatenate([nrm, view, alb, bump, col], 1).astype(np.float32)


def _outputs(H, W):
    return {"frame": torch.zeros((3, H, W), dtype=torch.uint8, device="cuda"),
            "depth": torch.ones((H, W), dtype=torch.float32, device="cuda")}


class _Slot:
    """A batch item's output buffer: a slice of a tensor the program owns."""

    def __init__(self, t):
        self.ptr = t.data_ptr()


SLOT_PIXELS = 1024 * 1024   # a batch item's share of the output tensors: the largest viewport


def _batch_work(case, seed):
    return scenes.batch_scenes(n=case["meshes"], seed=seed, max_faces=case["max_faces"])


_SHARED = []


def _context(case):
    """A program draws its meshes through one context; what is captured (a graph, the spin loop,
    an autotuned batch) belongs to a context of its own, as each would have in its own program."""
    if case.get("call") in ("graph", "spin"):
        return rz.Context(0)
    if not _SHARED:
        _SHARED.append(rz.Context(0))
    return _SHARED[0]


def prepare(case, seed):
    ctx = _context(case)
    s = {"case": case, "ctx": ctx}
    if case["kind"] == "train":
        data = _samples(case["samples"], seed)
        s.update(weights=_weights(seed), seed=seed)
        s["samples"] = rz.DeviceArray(ctx, data.shape, np.float32)
        s["samples"].upload(data)
    elif case["kind"] == "batch":
        work = _batch_work(case, seed)
        total = len(work) * SLOT_PIXELS
        s["out"] = {"frame": torch.zeros(3 * total, dtype=torch.uint8, device="cuda"),
                    "depth": torch.zeros(total, dtype=torch.float32, device="cuda")}
        if case["ids"]:
            s["out"]["ids"] = torch.zeros(total, dtype=torch.int32, device="cuda")
        s["items"] = []
        for (scene, args), o in zip(work, range(0, total, SLOT_PIXELS)):
            ids = _Slot(s["out"]["ids"][o:]) if case["ids"] else None
            s["items"].append((ctx.upload(scene), scene.lights_copy(), args, _Slot(s["out"]["frame"][3 * o:]),
                               _Slot(s["out"]["depth"][o:]), ids))
        torch.cuda.synchronize()
        if case["call"] == "graph":
            ctx.autotune(s["items"])
            s["graph"] = ctx.batch_graph(s["items"], 1)
    else:
        scene, args = _scene(case, seed)
        H, W = case["height"], case["width"]
        s.update(mesh=ctx.upload(scene), lights=scene.lights_copy(), args=args, flags=rz.RZ_FLAG_CLEARED, frame_no=0)
        if case["mlp"]:
            ctx.mlp_set_weights(_weights(1))   # the program's fitted network
            s["flags"] |= rz.RZ_FLAG_MLP_SHADE
        if case["call"] != "host":
            out = s["out"] = _outputs(H, W)
            ptrs = out["frame"].data_ptr(), out["depth"].data_ptr()
        torch.cuda.synchronize()
        if case["call"] == "graph":
            s["graph"] = ctx.graph(s["mesh"], s["lights"], args, *ptrs, case["frames"], flags=s["flags"], ry_step=0.01)
        elif case["call"] == "spin":
            s["spin"] = ctx.spin(s["mesh"], s["lights"], args, *ptrs)
        elif case["call"] == "overlay":
            second, args2 = _second(case, seed)
            out["ids"] = torch.zeros((H, W), dtype=torch.int32, device="cuda")
            s.update(mesh2=ctx.upload(second), lights2=second.lights_copy(), args2=args2)
    torch.cuda.synchronize()
    return s


# ---- a pass --------------------------------------------------------------------------


def run(state):
    s = state
    case, ctx = s["case"], s["ctx"]
    if case["kind"] == "train":
        ctx.mlp_set_weights(s["weights"])
        losses = ctx.mlp_train(s["samples"], case["samples"], case["steps"], case["batch"], 3e-3, s["seed"])
        return {"losses": losses, "weights": ctx.mlp_get_weights()}
    if case["kind"] == "batch":
        if case["call"] == "graph":
            s["graph"].launch()
            ctx.sync()
        else:
            ctx.draw_batch(s["items"])
        return s["out"]
    call = case["call"]
    if call == "host":
        frame, depth, _, _ = ctx.draw(s["mesh"], s["lights"], s["args"])
        return {"frame": frame, "depth": depth}
    out = s["out"]
    if call == "graph":
        s["graph"].launch()
        ctx.sync()
    elif call == "spin":
        a = s["args"].tait_bryan_angles
        s["spin"].frame((a[0], a[1] + 0.01 * s["frame_no"], a[2]))
        ctx.sync()   # the frame is shown before the next is drawn
        s["frame_no"] += 1
    else:
        ptrs = out["frame"].data_ptr(), out["depth"].data_ptr()
        flags = s["flags"] | (rz.RZ_FLAG_ASYNC if call != "device" else 0)
        ctx.draw_device(s["mesh"], s["lights"], s["args"], *ptrs, flags=flags)
        if call == "overlay":
            ctx.draw_device(s["mesh2"], s["lights2"], s["args2"], *ptrs, out["ids"].data_ptr(), flags=0)
    return out


# ---- what a pass cannot do without ----------------------------------------------------


def _mesh_size(case):
    """(faces, bytes of its faces' indices, positions, normals and uvs) of a frame case's mesh."""
    if case["mesh"] == "uv_sphere":
        return 960, 960 * 40 + 482 * 24
    if case["mesh"] == "icosphere":
        f = 20 * 4 ** case["detail"]
        return f, f * 40 + (f // 2 + 2) * 32
    return case["detail"], case["detail"] * (40 + 48)


def _batch_estimate(case):
    """(faces, pixels) a batch has on average: face counts log-uniform from 500, sides 256..1024."""
    faces = (case["max_faces"] - 500) / math.log(case["max_faces"] / 500)
    return case["meshes"] * faces, case["meshes"] * (640 ** 2 + 769 ** 2 / 12)


def work(case):
    if case["kind"] == "train":
        n = case["steps"] * case["batch"]
        return {"bytes": n * 60 + 2 * 4 * 5187, "flops": 3 * MLP_FLOPS * n}
    if case["kind"] == "batch":
        faces, pixels = _batch_estimate(case)
        return {"bytes": faces * (40 + 36) + pixels * (11 if case["ids"] else 7), "flops": 100 * faces + 60 * pixels}
    faces, mesh_bytes = _mesh_size(case)
    pixels = case["width"] * case["height"]
    per_frame = mesh_bytes + 4 * case["texture"] ** 2 * (2 if case["normal_map"] else 1) + 40 * case["lights"]
    frames = case.get("frames", 1)
    covered = 0.2 * pixels   # about what the meshes cover
    flops = 100 * faces + covered * (100 + (MLP_FLOPS if case["mlp"] else 12 * case["lights"]))
    nbytes = per_frame + 7 * pixels
    if case["call"] == "overlay":
        nbytes += per_frame + (14 + 4) * pixels
        flops *= 2
    return {"bytes": frames * nbytes, "flops": frames * flops}


# ---- 64-bit results -------------------------------------------------------------------


def _raster_vertices64(scene, args, frame_no):
    """The scene's vertices in raster space, (V, 3) float64: x, y in pixels, depth."""
    v = torch.from_numpy(scene.vertices).cuda().double()
    if scene.raster_space:
        return v[:, :3]
    ax, ay, az = (float(t) for t in args.tait_bryan_angles)
    ay += frame_no

    def rot(axis, t):
        c, s = math.cos(t), math.sin(t)
        i, j = ((1, 2), (2, 0), (0, 1))[axis]
        m = np.eye(3)
        m[i, i] = m[j, j] = c
        m[i, j], m[j, i] = -s, s
        return m

    R = torch.from_numpy(rot(1, ay) @ rot(0, ax) @ rot(2, az)).cuda()
    p = (v * float(args.scale)) @ R.T + torch.tensor(list(args.displacement), dtype=torch.float64, device="cuda")
    w = 3.0 - p[:, 2]
    f = 1.0 / math.tan(math.radians(float(args.fovy_degrees)) / 2)
    zn, zf = float(args.z_near), float(args.z_far)
    W, H = args.image_width, args.image_height
    x = 0.5 * (p[:, 0] * f / float(args.aspect_ratio) / w + 1) * W
    y = 0.5 * (1 - p[:, 1] * f / w) * H
    z = ((zf + zn) / (zf - zn) * w - 2 * zf * zn / (zf - zn)) / w
    return torch.stack([x, y, z], 1)


def _depth64(scene, args, depth=None, frame_no=0.0):
    """The frame's depth buffer (H * W) in 64-bit arithmetic, over `depth` or a cleared one."""
    W, H = args.image_width, args.image_height
    if depth is None:
        depth = torch.ones(H * W, dtype=torch.float64, device="cuda")
    p = _raster_vertices64(scene, args, frame_no)
    t = p[torch.from_numpy(scene.faces[:, :3].astype(np.int64)).cuda()]
    a, b, c = t[:, 0], t[:, 1], t[:, 2]

    def edge(q, r, x, y):
        return (r[:, 0] - q[:, 0]) * (y - q[:, 1]) - (r[:, 1] - q[:, 1]) * (x - q[:, 0])

    area = edge(c, a, b[:, 0], b[:, 1])
    twice = a[:, 0] * b[:, 1] - b[:, 0] * a[:, 1] + b[:, 0] * c[:, 1] - c[:, 0] * b[:, 1] + c[:, 0] * a[:, 1] - a[:, 0] * c[:, 1]
    front = (twice < 0) != bool(args.wind_clockwise)
    size = torch.tensor([W - 1.0, H - 1.0], dtype=torch.float64, device="cuda")
    lo = torch.minimum(t[:, :, :2].amin(1).clamp(min=0), size).floor().long()
    hi = torch.minimum(t[:, :, :2].amax(1).ceil().clamp(min=0), size).long()
    keep = front.nonzero()[:, 0]
    a, b, c, area, lo, hi = a[keep], b[keep], c[keep], area[keep], lo[keep], hi[keep]
    width = hi[:, 0] - lo[:, 0] + 1
    ends = torch.cumsum(width * (hi[:, 1] - lo[:, 1] + 1), 0)
    k = 0
    while k < len(ends):   # faces whose boxes hold about 2^24 pixels at a time
        begin = int(ends[k - 1]) if k else 0
        stop = max(k + 1, int(torch.searchsorted(ends, begin + (1 << 24))))
        count = ends[k:stop] - torch.cat([torch.tensor([begin], device="cuda"), ends[k:stop - 1]])
        f = torch.repeat_interleave(torch.arange(k, stop, device="cuda"), count)
        i = torch.arange(len(f), device="cuda") + begin - (ends[f] - count[f - k])
        x, y = lo[f, 0] + i % width[f], lo[f, 1] + i // width[f]
        A, B, C, xd, yd = a[f], b[f], c[f], x.double(), y.double()
        b0, b1, b2 = edge(B, C, xd, yd) / area[f], edge(C, A, xd, yd) / area[f], edge(A, B, xd, yd) / area[f]
        z = A[:, 2] * b0 + B[:, 2] * b1 + C[:, 2] * b2
        inside = (b0 >= 0) & (b1 >= 0) & (b2 >= 0)
        depth.scatter_reduce_(0, (y * W + x)[inside], z[inside], "amin")
        k = stop
    return depth


def _train64(case, seed):
    """The training burst in 64-bit arithmetic: losses and weights."""
    data = torch.from_numpy(_samples(case["samples"], seed)).cuda().double()
    p = torch.from_numpy(_weights(seed)).cuda().double()
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    n, losses = case["batch"], []
    for k in range(case["steps"]):
        with np.errstate(over="ignore"):   # the samples of a step: a hash of seed, step and place
            z = np.uint64(seed) + np.uint64(0x9E3779B97F4A7C15) * (np.uint64((k + 1) * 1048576 + 1) + np.arange(n, dtype=np.uint64))
            z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
            z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
            z = z ^ (z >> np.uint64(31))
        rows = data[torch.from_numpy((z % np.uint64(case["samples"])).astype(np.int64)).cuda()]
        w = p.clone().requires_grad_(True)
        parts, at = [], 0
        for s in MLP_LAYERS:
            parts.append(w[at:at + math.prod(s)].reshape(s))
            at += math.prod(s)
        W1, b1, W2, b2, W3, b3 = parts
        h = torch.relu(torch.relu(rows[:, :12] @ W1.T + b1) @ W2.T + b2)
        loss = (h @ W3.T + b3 - rows[:, 12:]).square().sum() / n
        loss.backward()
        losses.append(float(loss.detach()))
        lr = 3e-3 * (0.01 + 0.99 * 0.5 * (1 + math.cos(math.pi * k / case["steps"])))
        m, v = 0.9 * m + 0.1 * w.grad, 0.999 * v + 0.001 * w.grad ** 2
        p = p - lr * (m / (1 - 0.9 ** (k + 1))) / ((v / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    return {"losses": np.array(losses), "weights": p}


def exact(case, seed):
    if case["kind"] == "train":
        return _train64(case, seed)
    if case["kind"] == "batch":
        work_ = _batch_work(case, seed)
        depth = torch.zeros(len(work_) * SLOT_PIXELS, dtype=torch.float64, device="cuda")
        for k, (scene, args) in enumerate(work_):
            o, n = k * SLOT_PIXELS, args.image_width * args.image_height
            depth[o:o + n] = _depth64(scene, args)
        return {"frame": None, "depth": depth, "ids": None} if case["ids"] else {"frame": None, "depth": depth}
    scene, args = _scene(case, seed)
    turned = 0.01 * (case["frames"] - 1) if case["call"] == "graph" else 0.0
    depth = _depth64(scene, args, frame_no=turned)
    if case["call"] == "overlay":
        depth = _depth64(*_second(case, seed), depth=depth)
    depth = depth.reshape(case["height"], case["width"])
    return {"frame": None, "depth": depth, "ids": None} if case["call"] == "overlay" else {"frame": None, "depth": depth}
