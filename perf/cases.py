"""The work that a user of convector_amd has it do, as cases that can be timed
and whose outputs can be compared: ray queries, scene builds, rendering
(patches, frames, accumulations, batches, the request server) and the
denoiser (image and training step).

listed() names the fixed cases and draw() makes further ones of the same
ranges; prepare() makes a case's inputs from a seed, run() is one pass through
the public entry points, work() what a pass cannot do without, and exact() the
outputs in 64 bits where they are plain arithmetic.  A rendered image is the
result of millions of discrete branches (which triangle, which lobe, which
light), so it has no 64-bit value to compare with, and neither have the nodes
of a tree.
"""
from __future__ import annotations

import functools
import gzip
import math
import os
import tempfile

import numpy as np
import torch

import convector_amd as cv
from convector_amd import scenes

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# The denoiser's layers (cin, cout, level): the parameter vector holds
# [cout][3][3][cin] weights and cout biases per layer, the first layer's ten
# input channels padded to 16.
NET = [(16, 32, 0), (32, 32, 0), (32, 64, 1), (64, 64, 1), (64, 128, 2), (128, 128, 2),
       (192, 64, 1), (64, 64, 1), (96, 32, 0), (32, 32, 0), (32, 3, 0)]


def listed():
    return [
        # An editor's pick or a collision probe: a few rays, so the launches
        # and the wait are the cost.  suzanne: 968 triangles.
        dict(name="query-256-suzanne", kind="query", scene="suzanne", rays=256, coherent=False,
             full=False),
        # The reference's own intersect bench at a throughput size, ragged:
        # the bunny (69,666 triangles), nearest hits only.
        dict(name="query-10M-bunny", kind="query", scene="stanford_bunny", rays=10_000_019,
             coherent=False, full=False),
        # Full intersection records (position, normal, material, counters) of
        # rays inside a 200,000-triangle room, eight rays from one origin: what
        # a caller that shades by itself asks for.
        dict(name="query-1M-records-200k", kind="query", scene="room", tris=200_000,
             rays=1_000_003, coherent=True, full=True),
        # An interactive scene (20,506 triangles) loaded and its tree copied
        # out, as a program that bakes trees does.
        dict(name="build-20k", kind="build", tris=20_506, bins=64),
        # The same for the largest configuration.
        dict(name="build-1.33M", kind="build", tris=1_330_746, bins=64),
        # One 32 x 32 patch into the bitmap: the reference's unit of work.
        dict(name="patch-32", kind="patch", tris=20_506, width=1280, height=736, patch=32),
        # One interactive frame at the reference's window size, 1 sample,
        # bitmap and gbuffer on the host.
        dict(name="frame-1280x736", kind="frame", tris=20_506, width=1280, height=736),
        # Progressive accumulation of the largest configuration: 16 samples at
        # 1920 x 1080 over 1.33 M triangles into a device image.
        dict(name="accumulate-1080p-16spp", kind="accumulate", tris=1_330_746, width=1920,
             height=1080, spp=16),
        # A render farm's mix: 12 jobs of other scenes, sizes and sample counts
        # in shared launches, replayed as graphs.
        dict(name="batch-12-jobs", kind="batch", jobs=12, max_tris=200_000, max_width=1280,
             max_height=736, max_spp=8, pick=1000),
        # The request server under a burst: 16 requests over 3 resident scenes,
        # 256 x 256 to 1280 x 720, 1 to 4 samples, results to host memory.
        dict(name="serve-16-requests", kind="serve", requests=16, max_tris=200_000, max_spp=4,
             pick=2000),
        # A one-sample image at the window size denoised: features, network,
        # HDR image, on device buffers.
        dict(name="denoise-1280x736", kind="denoise", width=1280, height=736, spp=1),
        # One training step of the denoiser: 16 crops of 256 x 256, forward,
        # backward and Adam at the end of the learning rate's decay.
        dict(name="train-16x256", kind="train", batch=16, height=256, width=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, width, height, dx, dy):
    """A size up to width x height, a multiple of dx and dy."""
    return (max(dx, _log(rng, 64, width) // dx * dx), max(dy, _log(rng, 64, height) // dy * dy))


def draw(rng):
    kind = rng.choice(["query", "query", "build", "patch", "frame", "accumulate", "batch",
                       "serve", "denoise", "train"])
    if kind == "query":
        full = rng.random() < 0.4
        c = dict(kind=kind, scene=rng.choice(["suzanne", "stanford_bunny", "room"]),
                 rays=_log(rng, 64, 1 << 20 if full else 10_000_019),
                 coherent=rng.random() < 0.5, full=full)
        if c["scene"] == "room":
            c["tris"] = _log(rng, 1000, 200_000)
        return c
    if kind == "build":
        return dict(kind=kind, tris=_log(rng, 1000, 1_330_746), bins=rng.choice([64, 64, 32]))
    if kind == "patch":
        w, h = _size(rng, 1280, 736, 16, 16)
        return dict(kind=kind, tris=_log(rng, 1000, 20_506), width=w, height=h,
                    patch=rng.choice([16, 32]))
    if kind == "frame":
        w, h = _size(rng, 1280, 736, 16, 4)
        return dict(kind=kind, tris=_log(rng, 1000, 200_000), width=w, height=h)
    if kind == "accumulate":
        w, h = _size(rng, 1920, 1080, 16, 4)
        return dict(kind=kind, tris=_log(rng, 1000, 200_000), width=w, height=h,
                    spp=rng.randint(1, 16))
    if kind == "batch":
        return dict(kind=kind, jobs=rng.randint(2, 12), max_tris=_log(rng, 5000, 200_000),
                    max_width=1280, max_height=736, max_spp=rng.choice([1, 2, 4, 8]),
                    pick=rng.randint(1, 1 << 20))
    if kind == "serve":
        return dict(kind=kind, requests=rng.randint(1, 16), max_tris=_log(rng, 5000, 200_000),
                    max_spp=rng.choice([1, 2, 4]), pick=rng.randint(1, 1 << 20))
    if kind == "denoise":
        w, h = _size(rng, 1280, 736, 64, 4)
        return dict(kind=kind, width=w, height=h, spp=rng.choice([1, 2, 4]))
    return dict(kind=kind, batch=rng.randint(1, 16), height=_log(rng, 32, 256) // 4 * 4,
                width=64 * rng.randint(1, 4))


# ------------------------------------------------------------------ inputs


@functools.lru_cache(maxsize=None)
def _model(name):
    """A committed OBJ model, read by the library's loader."""
    src = os.path.join(ROOT, "tests", "golden", "models", name + ".obj.gz")
    with gzip.open(src, "rb") as f, tempfile.NamedTemporaryFile(suffix=".obj") as t:
        t.write(f.read())
        t.flush()
        return cv.Mesh.load(t.name)


@functools.lru_cache(maxsize=None)
def _ball(subdivisions):
    """Vertices and faces of the icosphere; the large ones displaced by smooth
    noise, as the largest configuration has it."""
    v, f = scenes.icosphere(subdivisions)
    if subdivisions >= 7:
        v = v * (0.4 + 0.08 * scenes.value_noise(v, 2))[:, None]
    return v, f


def _room(tris, seed):
    """A closed box with its light, a displaced sphere of as many faces as fit
    and free triangles for the rest."""
    k = 0
    while 20 * 4 ** (k + 1) <= tris - 26:
        k += 1
    st = scenes.Stream(seed)
    v, f = _ball(k)
    if k >= 7:  # the noise is fixed, so the seed turns the sphere
        a = float(st.uniform(1, 0.0, 2.0 * math.pi)[0])
        c, s = math.cos(a), math.sin(a)
        v = v @ np.array([[c, -s, 0.0], [s, c, 0.0], [0.0, 0.0, 1.0]])
    else:
        v = v * (0.4 + 0.05 * st.uniform(v.shape[0], -1.0, 1.0))[:, None]
    box, mats = scenes.box_with_light(scenes.Stream(seed ^ 0x5EED0B0C))
    parts = [box, np.concatenate([v[f[:, 0]], v[f[:, 1]], v[f[:, 2]]], 1)]
    mats = [mats, np.full(f.shape[0], scenes.MAT_GLOSSY_WHITE, np.uint32)]
    n = tris - 26 - f.shape[0]
    if n > 0:
        t, m = scenes.free_triangles(scenes.Stream(seed * 7919 + 17), n)
        parts.append(t)
        mats.append(m)
    t = np.concatenate(parts, 0).astype(np.float32)
    t[t == 0.0] = 0.0
    return scenes.SceneData(tris=t, materials=np.concatenate(mats).astype(np.uint32),
                            emission_override=(10.0, 10.0, 10.0))


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _sphere_points(n, g):
    p = torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float64)
    return p / p.norm(dim=1, keepdim=True)


def _rays(case, seed):
    """Rays from a sphere toward points of a smaller one: from outside the
    model, or inside the room; coherent: one origin for eight rays."""
    n, g = case["rays"], _generator(seed)
    radius, target = (0.9, 0.6) if case["scene"] == "room" else (10.0, 1.0)
    if case["coherent"]:
        o = _sphere_points((n + 7) // 8, g).repeat_interleave(8, 0)[:n] * radius
        d = _sphere_points(n, g) * (0.5 * target)
    else:
        o = _sphere_points(n, g) * radius
        d = _sphere_points(n, g) * target
    d = d - o
    d = d / d.norm(dim=1, keepdim=True)
    return torch.cat([o, d], 1).float().contiguous()


def _mix(case):
    """(triangles, seed, width, height, samples) of a batch's jobs."""
    return scenes.batch_jobs(case["jobs"], seed0=case["pick"],
                             tri_range=(1e3, float(case["max_tris"])),
                             width_range=(64, case["max_width"]),
                             height_range=(64, case["max_height"]), max_spp=case["max_spp"])


def _requests(case):
    """(scene, width, height, samples, camera x, camera z) of a burst."""
    st, out = scenes.Stream(case["pick"]), []
    for _ in range(case["requests"]):
        u = st.uniform(5, 0.0, 1.0)
        w, h = ((256, 256), (640, 368), (1280, 720))[min(int(3 * u[1]), 2)]
        spp = 1 << int(u[2] * (math.log2(case["max_spp"]) + 1 - 1e-9))
        out.append((min(int(3 * u[0]), 2), w, h, spp, 0.6 * u[3] - 0.3, 0.6 * u[4] - 0.3))
    return out


def _serve_tris(case):
    """Triangles of the three resident scenes."""
    return [1000, int(math.sqrt(1000.0 * case["max_tris"])), case["max_tris"]]


def _params(g):
    """He-normal weights and small biases in the flat order."""
    parts = []
    for cin, cout, _ in NET:
        std = math.sqrt(2.0 / (9 * cin))
        parts.append(std * torch.randn(cout * 9 * cin, generator=g, device="cuda"))
        parts.append(0.02 * torch.randn(cout, generator=g, device="cuda"))
    return torch.cat(parts).float()


def _radiance(shape, g):
    """Noisy one-sample radiance: dark with bright outliers."""
    r = torch.randn(shape, generator=g, device="cuda")
    return torch.exp(1.3 * r - 1.0) * (torch.rand(shape, generator=g, device="cuda") < 0.7)


def _features(n, spp, g):
    """First-hit features summed over spp samples: albedo, normal, distance,
    count."""
    f = torch.empty((n, 8), device="cuda")
    f[:, 0:3] = 0.2 + 0.6 * torch.rand((n, 3), generator=g, device="cuda")
    m = torch.randn((n, 3), generator=g, device="cuda")
    f[:, 3:6] = m / m.norm(dim=1, keepdim=True)
    f[:, 6] = 0.3 + 1.7 * torch.rand(n, generator=g, device="cuda")
    f[:, 7] = 1.0
    return (f * float(spp)).contiguous()


def _net_inputs(case, seed):
    """Parameters and device inputs of the denoiser's cases."""
    g = _generator(seed)
    p = _params(g)
    if case["kind"] == "denoise":
        n = case["width"] * case["height"]
        return p, _radiance((n * 3,), g) * float(case["spp"]), _features(n, case["spp"], g)
    shape = (case["batch"], case["height"], case["width"])
    x = torch.empty(shape + (10,), device="cuda")
    x[..., 0:3] = torch.log1p(_radiance(shape + (3,), g))
    x[..., 3:6] = 0.2 + 0.6 * torch.rand(shape + (3,), generator=g, device="cuda")
    x[..., 6:8] = 2.0 * torch.rand(shape + (2,), generator=g, device="cuda") - 1.0
    x[..., 8] = torch.log1p(0.3 + 1.7 * torch.rand(shape, generator=g, device="cuda"))
    x[..., 9] = 1.0
    target = torch.exp(0.8 * torch.randn(shape + (3,), generator=g, device="cuda") - 1.0)
    return p, x.contiguous(), target.contiguous()


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "query":
        if case["scene"] == "room":
            s["scene"] = cv.Scene.from_scene_data(_room(case["tris"], seed))
        else:
            s["scene"] = cv.Scene.from_meshes([_model(case["scene"])])
        n = case["rays"]
        s["rays"] = _rays(case, seed)
        s["hits"] = torch.zeros((n, 4), device="cuda", dtype=torch.int32)
        s["records"] = (torch.zeros((n, 16), device="cuda", dtype=torch.int32)
                        if case["full"] else None)
    elif kind == "build":
        sd = _room(case["tris"], seed)
        s["mesh"] = cv.Mesh.from_triangles(sd.tris, sd.materials)
        # a tree has at most two nodes per triangle, and a pair
        s["nodes"] = np.zeros(2 * sd.ntris + 2, cv.NODE_DTYPE)
        s["order"] = np.zeros(sd.ntris, np.uint32)
    elif kind in ("patch", "frame", "accumulate"):
        s["scene"] = cv.Scene.from_scene_data(_room(case["tris"], seed))
        s["renderer"] = cv.Renderer(s["scene"], case["width"], case["height"])
        s["frame"] = 1 + seed % 1000
        n = case["width"] * case["height"]
        if kind == "patch":
            s["bitmap"], s["gbuffer"] = s["renderer"].new_bitmap(), s["renderer"].new_bitmap()
            s["patch"] = seed
        elif kind == "accumulate":
            s["hdr"] = torch.zeros(n * 3, device="cuda")
    elif kind == "batch":
        s["jobs"], s["hdr"] = [], []
        for k, (tris, _, w, h, spp) in enumerate(_mix(case)):
            hdr = torch.zeros(w * h * 3, device="cuda")
            s["hdr"].append(hdr)
            s["jobs"].append(cv.Job(cv.Scene.from_scene_data(_room(tris, seed + k)), w, h, 1, spp,
                                    hdr=hdr.data_ptr()))
        s["batch"] = cv.Batch()
    elif kind == "serve":
        s["server"] = cv.Server()
        s["ids"] = [s["server"].add_scene(cv.Scene.from_scene_data(_room(t, seed + k)))
                    for k, t in enumerate(_serve_tris(case))]
        s["requests"] = [r + (np.zeros(r[1] * r[2] * 3, np.float32),) for r in _requests(case)]
    else:
        s["net"] = cv.Denoiser(1)
        p, a, b = _net_inputs(case, seed)
        s["net"].set_params(p.cpu().numpy())
        if kind == "denoise":
            n = case["width"] * case["height"]
            s["noisy"], s["features"] = a, b
            s["input"] = torch.zeros((n, 10), device="cuda")
            s["output"] = torch.zeros((n, 3), device="cuda")
            s["hdr"] = torch.zeros(n * 3, device="cuda")
        else:
            s["input"], s["target"] = a, b
    return s


# --------------------------------------------------------------------- run


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "query":
        hits, records = s["hits"], s["records"]
        s["scene"].intersect_nearest_device(s["rays"].data_ptr(), case["rays"], hits.data_ptr(),
                                            records.data_ptr() if records is not None else None)
        out = {"tri": hits[:, 0], "t": hits.view(torch.float32)[:, 1], "uv": hits[:, 2:]}
        return out if records is None else dict(out, records=records)
    if kind == "build":
        scene = cv.Scene.from_meshes([s["mesh"]], bins=case["bins"])
        cv.check(cv.lib().cv_scene_copy_bvh(scene._h, s["nodes"].ctypes.data,
                                            s["order"].ctypes.data))
        return {"info": [scene.bvh_info()[k] for k in ("num_nodes", "depth", "max_leaf")],
                "nodes": s["nodes"].view(np.int32), "order": s["order"].view(np.int32)}
    if kind == "patch":
        pw = case["patch"]
        across, up = case["width"] // pw, case["height"] // pw
        k = s["patch"] % (across * up)
        s["patch"] += 1
        s["renderer"].render_patch_u8(s["bitmap"], s["gbuffer"], pw, k % across * pw,
                                      k // across * pw, s["frame"])
        return {"bitmap": s["bitmap"].view(np.int32), "gbuffer": s["gbuffer"].view(np.int32)}
    if kind == "frame":
        s["frame"] += 1
        bitmap, gbuffer = s["renderer"].render_frame_u8(s["frame"])
        return {"bitmap": bitmap.view(np.int32), "gbuffer": gbuffer.view(np.int32)}
    if kind == "accumulate":
        s["renderer"].accumulate_frames_device(s["hdr"].data_ptr(), s["frame"], case["spp"])
        s["frame"] += case["spp"]
        return s["hdr"]
    if kind == "batch":
        s["batch"].render(s["jobs"], cv.PTR_DEVICE | cv.RENDER_GRAPH)
        return s["hdr"]
    if kind == "serve":
        tickets = [s["server"].submit(s["ids"][r[0]], r[1], r[2], r[3], (r[4], 0.9, r[5]),
                                      (0.70710677, -0.70710677, 0.0, 0.0), hdr=r[6])[0]
                   for r in s["requests"]]
        for t in tickets:
            s["server"].wait(t)
        return [r[6] for r in s["requests"]]
    net, w, h = s["net"], case["width"], case["height"]
    if kind == "denoise":
        net.prepare_input_device(s["noisy"].data_ptr(), s["features"].data_ptr(), w, h,
                                 case["spp"], s["input"].data_ptr())
        net.forward_device(s["input"].data_ptr(), s["output"].data_ptr(), 1, h, w)
        cv.check(cv.lib().cv_denoiser_output_to_hdr(s["output"].data_ptr(), w, h, case["spp"],
                                                    s["hdr"].data_ptr(), cv.PTR_DEVICE))
        return {"input": s["input"], "output": s["output"], "hdr": s["hdr"]}
    loss = net.train_step_device(s["input"].data_ptr(), s["target"].data_ptr(), case["batch"], h,
                                 w, 1e-6)
    return {"loss": loss, "grads": net.grads(), "params": net.params()}


# -------------------------------------------------------------------- work


def _tree(tris):
    """Bytes of a scene's tree and triangles, each read once: two 32-byte
    nodes and 48 bytes of vertices and edges per triangle."""
    return 112 * tris


def _query_flops(tris, inside):
    """Box and triangle tests of one nearest hit (23 and 48 operations each)
    by the reference's traversal, as its counters grow with the tree's depth:
    about 2.5 boxes a level for rays from outside a model and 6.5 inside a
    closed room."""
    return 23 * (6.5 if inside else 2.5) * math.log2(tris) + 48 * (4.8 if inside else 2.3)


def _render(paths, tris):
    """Operations of camera paths of up to five bounces: 4.5 queries each with
    8 light tests and the shading of a hit (about 470)."""
    return paths * 4.5 * (_query_flops(tris, True) + 470)


def _net_flops(pixels):
    return sum(2 * 9 * (10 if i == 0 else cin) * cout * (pixels >> (2 * level))
               for i, (cin, cout, level) in enumerate(NET))


def work(case):
    kind = case["kind"]
    if kind == "query":
        tris = {"suzanne": 968, "stanford_bunny": 69_666}.get(case["scene"]) or case["tris"]
        return {"bytes": case["rays"] * (24 + 16 + (64 if case["full"] else 0)) + _tree(tris),
                "flops": case["rays"] * _query_flops(tris, case["scene"] == "room")}
    if kind == "build":
        # triangles and materials in; nodes, order and the traversal's triangles out
        n = case["tris"]
        return {"bytes": n * (36 + 24 + 4) + _tree(n) + n * (4 + 4 + 24),
                "flops": n * math.log2(n) * 3 * 10}
    if kind == "patch":
        n = case["patch"] ** 2
        return {"bytes": 8 * n + min(_tree(case["tris"]), 4096 * n), "flops": _render(n, case["tris"])}
    if kind in ("frame", "accumulate"):
        n, spp = case["width"] * case["height"], case.get("spp", 1)
        return {"bytes": n * (8 if kind == "frame" else 24) + _tree(case["tris"]),
                "flops": _render(n * spp, case["tris"])}
    if kind == "batch":
        m = _mix(case)
        return {"bytes": sum(24 * w * h + _tree(t) for t, _, w, h, _ in m),
                "flops": sum(_render(w * h * spp, t) for t, _, w, h, spp in m)}
    if kind == "serve":
        t = _serve_tris(case)
        return {"bytes": sum(_tree(x) for x in t) + sum(12 * r[1] * r[2] for r in _requests(case)),
                "flops": sum(_render(r[1] * r[2] * r[3], t[r[0]]) for r in _requests(case))}
    if kind == "denoise":
        n = case["width"] * case["height"]
        return {"bytes": n * (12 + 32 + 40 + 12 + 12), "flops": _net_flops(n)}
    n, p = case["batch"] * case["height"] * case["width"], sum(9 * a * b + b for a, b, _ in NET)
    # forward, and twice its products backward but for the first layer's input
    return {"bytes": n * (40 + 12) + p * 4 * 8,
            "flops": 3 * _net_flops(n) - 2 * 9 * 10 * 32 * n}


# ------------------------------------------------------------------- exact


def _nearest(rays, tris):
    """Distance of each ray's nearest hit by brute force (1e5: none)."""
    o, d = rays[:, None, 0:3], rays[:, None, 3:6]
    best = torch.full((rays.shape[0],), 1e5, device="cuda", dtype=torch.float64)
    for part in tris.split(max(1, 20_000_000 // rays.shape[0])):
        v0, v1, v2 = part[None, :, 0:3], part[None, :, 3:6], part[None, :, 6:9]
        e1, e2 = v1 - v0, v2 - v0
        p = torch.linalg.cross(d, e2.expand(rays.shape[0], -1, -1))
        det = (p * e1).sum(-1)
        s = o - v0
        u = (s * p).sum(-1) / det
        q = torch.linalg.cross(s, e1.expand(rays.shape[0], -1, -1))
        v = (d * q).sum(-1) / det
        t = (e2 * q).sum(-1) / det
        ok = (u >= 0) & (v >= 0) & (u + v <= 1) & (t > 0)
        best = torch.minimum(best, torch.where(ok, t, best[:, None]).amin(1))
    return best


def _conv(x, w, b):
    """3 x 3 convolution of (n, h, w, cin) by [cout][3][3][cin] weights."""
    n, h, wd, _ = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    y = b
    for ky in range(3):
        for kx in range(3):
            y = y + xp[:, ky:ky + h, kx:kx + wd, :].contiguous() @ w[:, ky, kx, :].t().contiguous()
    return y


def _network(x, p):
    """The denoiser in the precision of its arguments; x: (n, h, w, 10)."""
    x = torch.nn.functional.pad(x, (0, 6))
    wb, at = [], 0
    for cin, cout, _ in NET:
        wb.append((p[at:at + 9 * cin * cout].view(cout, 3, 3, cin),
                   p[at + 9 * cin * cout:at + 9 * cin * cout + cout]))
        at += 9 * cin * cout + cout

    def layer(t, k):
        return torch.relu(_conv(t, *wb[k]))

    def pool(t):
        return (t[:, 0::2, 0::2] + t[:, 0::2, 1::2] + t[:, 1::2, 0::2] + t[:, 1::2, 1::2]) / 4

    def up(t):
        return t.repeat_interleave(2, 1).repeat_interleave(2, 2)

    e0 = layer(layer(x, 0), 1)
    e1 = layer(layer(pool(e0), 2), 3)
    b2 = layer(layer(pool(e1), 4), 5)
    d1 = layer(layer(torch.cat([up(b2), e1], 3), 6), 7)
    d0 = layer(layer(torch.cat([up(d1), e0], 3), 8), 9)
    return _conv(d0, *wb[10])


def _blocks(image):
    """(h, w, 3) as the HDR layout: 16 x 4 blocks of [8 groups][3][8 lanes]; a
    group is 4 pixels wide and 2 high, the lower of two groups first."""
    h, w, _ = image.shape
    b = image.view(h // 4, 2, 2, w // 16, 4, 4, 3)  # block row, group, y, block, group, x
    return b.permute(0, 3, 4, 1, 6, 2, 5).reshape(-1)


def _image(hdr, w, h):
    """The inverse of _blocks."""
    b = hdr.view(h // 4, w // 16, 4, 2, 3, 2, 4)
    return b.permute(0, 3, 5, 1, 2, 6, 4).reshape(h, w, 3)


def exact(case, seed):
    kind = case["kind"]
    if kind == "query":
        if case["scene"] == "room":
            tris = _room(case["tris"], seed).tris
        else:
            tris = _model(case["scene"]).triangles()[0]
        if case["rays"] * len(tris) > 1_000_000_000:
            return None
        tris = torch.from_numpy(np.ascontiguousarray(tris)).cuda().double()
        out = {"tri": None, "t": _nearest(_rays(case, seed).double(), tris), "uv": None}
        return dict(out, records=None) if case["full"] else out
    if kind not in ("denoise", "train"):
        return None
    p, a, b = (t.double() for t in _net_inputs(case, seed))
    if kind == "denoise":
        w, h, spp = case["width"], case["height"], case["spp"]
        f = b / spp
        n = f[:, 3:6] / f[:, 3:6].abs().sum(1, keepdim=True)
        sign = torch.where(n[:, 0:2] >= 0, 1.0, -1.0).double()
        fold = (1.0 - n[:, 0:2].abs().flip(1)) * sign
        n = torch.where(n[:, 2:3] < 0, fold, n[:, 0:2])
        x = torch.cat([torch.log1p(_image(a, w, h).reshape(-1, 3) / spp), f[:, 0:3], n,
                       torch.log1p(f[:, 6:7]), torch.full_like(f[:, 6:7], spp)], 1)
        y = _network(x.view(1, h, w, 10), p)
        hdr = _blocks(torch.expm1(y[0].clamp(min=0.0)) * spp)
        return {"input": x, "output": y.view(-1, 3), "hdr": hdr}
    p.requires_grad_(True)
    loss = (_network(a, p) - torch.log1p(b)).abs().mean()
    loss.backward()
    # Adam's first step from zero moments: lr g / (|g| + eps) after its bias correction
    with torch.no_grad():
        new = p - 1e-6 * p.grad / (p.grad.abs() + 1e-8)
    return {"loss": float(loss), "grads": p.grad.cpu().numpy(), "params": new.cpu().numpy()}
