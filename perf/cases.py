"""The work that users of xtracer_amd have it do, as cases that can be timed.

A program that uses this package keeps one device handle with its scenes
resident and then makes four kinds of calls on it:

  trace   closest-hit queries on device-resident rays (`Device.trace_device`)
  render  one job into a device framebuffer (`Device.render_device`)
  serve   a batch of jobs through the continuous-batching server
          (`Device.submit` / `drain` / `poll`)
  admit   a new scene made resident, its first frame rendered, and released

A case names one such call with its scene and sizes. The scenes are the
package's seeded generators (64 spheres on a plane, displaced icosphere,
terrain, hair strands); the seed of `prepare` draws the camera pose, the rays
and the random streams, which is what differs from call to call. The device
handle and the loaded scenes are kept for the life of the process, as such a
program keeps them; `admit` pays for residency inside the call.
"""
import math
import os

import numpy as np
import torch

import xtracer_amd as xa
from xtracer_amd import scenes

# scene name -> (generator, its arguments, camera, box that random rays start in)
_SCENES = {
    "spheres": (scenes.spheres, {}, scenes.SPHERES_CAMERA, ((-2.0, 0.2, -4.0), (12.0, 10.0, 12.0))),
    "ico5": (scenes.icosphere_scene, {"subdiv": 5}, scenes.ICOSPHERE_CAMERA, ((-2.5, 0.1, -2.5), (2.5, 3.1, 2.5))),
    "ico7": (scenes.icosphere_scene, {"subdiv": 7}, scenes.ICOSPHERE_CAMERA, ((-2.5, 0.1, -2.5), (2.5, 3.1, 2.5))),
    "ico8": (scenes.icosphere_scene, {"subdiv": 8}, scenes.ICOSPHERE_CAMERA, ((-2.5, 0.1, -2.5), (2.5, 3.1, 2.5))),
    "terrain": (scenes.terrain_scene, {}, scenes.TERRAIN_CAMERA, ((-3.5, 0.8, -3.5), (3.5, 3.0, 3.5))),
    "terrain41": (scenes.terrain_scene, {"n": 41}, scenes.TERRAIN_CAMERA, ((-3.5, 0.8, -3.5), (3.5, 3.0, 3.5))),
    "strands": (scenes.strands_scene, {"strands": 50000}, scenes.STRANDS_CAMERA, ((-1.2, -1.2, -1.2), (1.2, 1.2, 1.2))),
}
# triangles (and spheres) of each scene, for the work estimates
_PRIMS = {"spheres": 65, "ico5": 20493, "ico7": 327693, "ico8": 1310733, "terrain": 199713, "terrain41": 3201,
          "strands": 2950012}
# mean closest-hit queries per camera sample
_QUERIES = {"stencil": 1.0, "depth": 1.0, "normal": 1.0, "ao": 1.6, "pathtracer": 2.2}

_kept = {}


def _device():
    if "device" not in _kept:
        _kept["device"] = xa.Device(0)
    return _kept["device"]


def _path(name):
    fn, kw, _, _ = _SCENES[name]
    return fn(**kw)


def _host_scene(name, on_device):
    key = ("host", name, on_device)
    if key not in _kept:
        _kept[key] = xa.Scene(_path(name), kd_on_device=on_device)
    return _kept[key]


def _scene_id(name):
    key = ("sid", name)
    if key not in _kept:
        _kept[key] = _device().upload(_host_scene(name, False))
    return _kept[key]


def _pose(name, seed):
    """The scene camera moved to a random place on the sphere through it
    around its target, as serving requests with views of their own do."""
    cam = _SCENES[name][2]
    rng = np.random.default_rng([seed, 11])
    p, t = np.asarray(cam["position"], float), np.asarray(cam["target"], float)
    r = float(np.linalg.norm(p - t))
    az, el = rng.uniform(0, 2 * np.pi), rng.uniform(0.05, 0.6)
    pos = t + r * np.array([np.cos(el) * np.sin(az), np.sin(el), np.cos(el) * np.cos(az)])
    return {"position": [float(np.float32(c)) for c in pos], "target": [float(np.float32(c)) for c in t],
            "fov": cam.get("fov", 45.0), "aperture": cam.get("aperture", 0.0), "flength": cam.get("flength", 0.0)}


def _camera(pose):
    return xa.make_camera(pose["position"], pose["target"], (0.0, 1.0, 0.0), pose["fov"], pose["aperture"],
                          pose["flength"])


def _rays(name, n, how, seed):
    """(n, 4) origin and direction records in FP32 on the GPU, origin word
    "free ray". "random": from anywhere around the scene in any direction, as
    visibility probes are; "camera": a pinhole's rays over a square image."""
    g = torch.Generator(device="cuda").manual_seed(1000003 * (seed + 1) + n)
    if how == "camera":
        pose = _pose(name, seed)
        pos = torch.tensor(pose["position"], dtype=torch.float64, device="cuda")
        z = torch.tensor(pose["target"], dtype=torch.float64, device="cuda") - pos
        z = z / z.norm()
        x = torch.linalg.cross(torch.tensor([0.0, 1.0, 0.0], dtype=torch.float64, device="cuda"), z)
        x = x / x.norm()
        y = torch.linalg.cross(z, x)
        side = max(1, int(math.isqrt(n - 1)) + 1)
        i = torch.arange(n, device="cuda")
        s = math.tan(math.radians(pose["fov"]) / 2)
        jit = torch.rand((n, 2), generator=g, device="cuda", dtype=torch.float64)
        px = (((i % side) + jit[:, 0]) / side * 2 - 1) * s
        py = ((torch.div(i, side, rounding_mode="floor") + jit[:, 1]) / side * 2 - 1) * s
        d = z + px[:, None] * x + py[:, None] * y
        o = pos.expand(n, 3)
    else:
        lo, hi = (torch.tensor(v, dtype=torch.float64, device="cuda") for v in _SCENES[name][3])
        o = lo + (hi - lo) * torch.rand((n, 3), generator=g, device="cuda", dtype=torch.float64)
        d = torch.randn((n, 3), generator=g, device="cuda", dtype=torch.float64)
    d = d / d.norm(dim=1, keepdim=True)
    r0 = torch.empty((n, 4), dtype=torch.float32, device="cuda")
    r1 = torch.zeros((n, 4), dtype=torch.float32, device="cuda")
    r0[:, :3] = o
    r0.view(torch.int32)[:, 3] = -1
    r1[:, :3] = d
    return r0, r1


def listed():
    return [
        # a picking or visibility program's single call: latency is all that counts
        {"name": "trace_64_spheres", "kind": "trace", "scene": "spheres", "rays": 64, "how": "random"},
        # probe rays of an ordinary batch, an odd number of them
        {"name": "trace_100003_terrain", "kind": "trace", "scene": "terrain", "rays": 100003, "how": "random"},
        # a large batch of incoherent queries against a large mesh
        {"name": "trace_4m_icosphere", "kind": "trace", "scene": "ico8", "rays": 1 << 22, "how": "random"},
        # an editor's thumbnail
        {"name": "stencil_33x17_spheres", "kind": "render", "scene": "spheres", "integrator": "stencil", "width": 33,
         "height": 17, "spp": 1, "rdepth": 1},
        # an editor's depth preview at a ragged size
        {"name": "depth_333x211_terrain", "kind": "render", "scene": "terrain", "integrator": "depth", "width": 333,
         "height": 211, "spp": 1, "rdepth": 1},
        # a normal buffer for a compositor, odd in both directions
        {"name": "normal_1001x701_icosphere", "kind": "render", "scene": "ico7", "integrator": "normal",
         "width": 1001, "height": 701, "spp": 2, "rdepth": 1},
        # ambient occlusion, the serving mix's sphere jobs
        {"name": "ao_512x512x16_spheres", "kind": "render", "scene": "spheres", "integrator": "ao", "width": 512,
         "height": 512, "spp": 16, "rdepth": 1},
        # an interactive path-traced refresh
        {"name": "path_256x256x4_terrain", "kind": "render", "scene": "terrain", "integrator": "pathtracer",
         "width": 256, "height": 256, "spp": 4, "rdepth": 8},
        # the benchmark's hair workload at a quarter of its samples
        {"name": "path_1024x1024x8_strands", "kind": "render", "scene": "strands", "integrator": "pathtracer",
         "width": 1024, "height": 1024, "spp": 8, "rdepth": 6},
        # the benchmark's frame: 1.31 M triangles, 33.2 M paths
        {"name": "path_1080p16_icosphere", "kind": "render", "scene": "ico8", "integrator": "pathtracer",
         "width": 1920, "height": 1080, "spp": 16, "rdepth": 8},
        # a batch of mixed jobs through the server
        {"name": "serve_16_jobs", "kind": "serve", "jobs": 16, "mix": 1, "most": 512},
        # a new scene: upload, tree build, first depth frame, release
        {"name": "admit_terrain", "kind": "admit", "scene": "terrain", "width": 512, "height": 384},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["trace", "render", "serve", "admit"], [7, 10, 1, 2])[0]
    if kind == "trace":
        scene = rng.choice(["spheres", "ico5", "ico7", "ico8", "terrain", "terrain41", "strands"])
        return {"kind": "trace", "scene": scene, "rays": _log_int(rng, 48, 1 << 22),
                "how": rng.choice(["random", "camera"])}
    if kind == "render":
        scene = rng.choice(["spheres", "ico5", "ico7", "ico8", "terrain", "terrain41", "strands"])
        integrator = rng.choice(["pathtracer", "pathtracer", "pathtracer", "ao", "ao", "depth", "normal", "stencil"])
        pixels = _log_int(rng, 400, 1 << 20)
        aspect = rng.uniform(0.6, 1.9)
        width = max(9, int(math.sqrt(pixels * aspect)))
        height = max(9, pixels // width)
        return {"kind": "render", "scene": scene, "integrator": integrator, "width": width, "height": height,
                "spp": rng.choice([1, 2, 3, 4, 8, 16]) if integrator in ("pathtracer", "ao") else rng.choice([1, 2, 4]),
                "rdepth": rng.randint(2, 8) if integrator == "pathtracer" else 1}
    if kind == "serve":
        return {"kind": "serve", "jobs": rng.randint(3, 16), "mix": rng.randrange(1, 1 << 20),
                "most": rng.choice([128, 256, 512])}
    return {"kind": "admit", "scene": rng.choice(["spheres", "ico5", "terrain", "terrain41"]),
            "width": rng.randint(64, 512), "height": rng.randint(48, 384)}


# scene, integrator and depth of the server's jobs
_SERVED = [("spheres", "ao", 1), ("ico7", "pathtracer", 8), ("terrain", "pathtracer", 8)]


def _mix(case):
    """The batch's jobs: scene, integrator, depth, edge length and samples of each."""
    rng = np.random.default_rng(case["mix"])
    sizes = [s for s in (128, 200, 256, 333, 512) if s <= case["most"]]
    return [(*_SERVED[int(rng.integers(len(_SERVED)))], int(rng.choice(sizes)), int(rng.choice([1, 4, 16])))
            for _ in range(case["jobs"])]


def prepare(case, seed):
    dev = _device()
    st = {"kind": case["kind"], "dev": dev}
    if case["kind"] == "trace":
        st["sid"] = _scene_id(case["scene"])
        st["n"] = case["rays"]
        st["r0"], st["r1"] = _rays(case["scene"], case["rays"], case["how"], seed)
        st["hit"] = torch.zeros((case["rays"], 4), dtype=torch.float32, device="cuda")
    elif case["kind"] == "serve":
        st["jobs"] = []
        for k, (scene, integrator, rdepth, res, spp) in enumerate(_mix(case)):
            cam = _camera(_pose(scene, 1000 * seed + k))
            st["jobs"].append(xa.make_job(_scene_id(scene), integrator, res, res, cam, samples=spp, rdepth=rdepth,
                                          seed=seed + 1, job_key=k))
    else:
        cam = _camera(_pose(case["scene"], seed))
        st["out"] = torch.zeros((case["height"], case["width"], 4), dtype=torch.float32, device="cuda")
        if case["kind"] == "admit":
            st["scene"] = _host_scene(case["scene"], True)
            st["job"] = xa.make_job(0, "depth", case["width"], case["height"], cam, seed=seed + 1)
        else:
            st["job"] = xa.make_job(_scene_id(case["scene"]), case["integrator"], case["width"], case["height"], cam,
                                    samples=case["spp"], rdepth=case["rdepth"], seed=seed + 1)
    # the library works on streams of its own: what torch has queued ends here
    torch.cuda.synchronize()
    return st


def run(state):
    dev = state["dev"]
    if state["kind"] == "trace":
        dev.trace_device(state["sid"], state["r0"].data_ptr(), state["r1"].data_ptr(), state["hit"].data_ptr(),
                         state["n"])
        hit = state["hit"]
        return {"t": hit[:, 0], "prim": hit.view(torch.int32)[:, 1], "u": hit[:, 2], "v": hit[:, 3]}
    if state["kind"] == "render":
        dev.render_device(state["job"], state["out"].data_ptr())
        return state["out"]
    if state["kind"] == "serve":
        tickets = [dev.submit(j) for j in state["jobs"]]
        dev.drain()
        return [dev.poll(t, j.width, j.height)[1] for t, j in zip(tickets, state["jobs"])]
    sid = dev.upload(state["scene"])
    state["job"].scene_id = sid
    dev.render_device(state["job"], state["out"].data_ptr())
    dev.release(sid)
    return state["out"]


def _query_work(scene, queries):
    """Rays read (32 B) and hits written (16 B); the triangles that the
    queries can need, once (36 B); two boxes for each level of a balanced
    tree (18 operations a box) and two triangle tests (50)."""
    n = _PRIMS[scene]
    return {"bytes": 48.0 * queries + 36.0 * min(n, 4 * queries),
            "flops": queries * (36.0 * math.log2(n) + 100.0)}


def work(case):
    if case["kind"] == "trace":
        return _query_work(case["scene"], case["rays"])
    if case["kind"] == "serve":
        total = {"bytes": 0.0, "flops": 0.0}
        for scene, integrator, _, res, spp in _mix(case):
            w = _query_work(scene, res * res * spp * _QUERIES[integrator])
            total["bytes"] += w["bytes"] + 16.0 * res * res
            total["flops"] += w["flops"]
        return total
    pixels = case["width"] * case["height"]
    if case["kind"] == "admit":
        # per primitive its FP32 and FP64 records, texture coordinates and
        # octree item in, a tree of about as many nodes out
        n = _PRIMS[case["scene"]]
        w = _query_work(case["scene"], pixels)
        return {"bytes": w["bytes"] + n * (48.0 + 72.0 + 48.0 + 4.0 + 16.0) + 16.0 * pixels,
                "flops": w["flops"] + n * 100.0 * math.log2(n)}
    w = _query_work(case["scene"], pixels * case["spp"] * _QUERIES[case["integrator"]])
    return {"bytes": w["bytes"] + 16.0 * pixels, "flops": w["flops"]}


# ------------------------------------------------------------------ 64 bits

def _obj_triangles(path):
    """(n, 9) corners of an OBJ file of `v` lines followed by triangle `f` lines."""
    with open(path) as f:
        text = f.read()
    at = text.index("\nf ") + 1
    head = text[text.index("v "):at]
    v = np.array(head.replace("v", " ").split(), dtype=np.float32).astype(np.float64).reshape(-1, 3)
    f = np.array(text[at:].replace("f", " ").split(), dtype=np.int64).reshape(-1, 3) - 1
    return v[f].reshape(-1, 9)


def _geometry(name):
    """(triangles (n, 9), spheres (n, 4), whether there is the floor y = 0) of a scene, from its files."""
    key = ("exact", name)
    if key not in _kept:
        path = _path(name)
        d = os.path.dirname(path)
        tris = [_obj_triangles(os.path.join(d, f)) for f in sorted(os.listdir(d)) if f.endswith(".obj")]
        balls = []
        with open(path) as f:
            for part in f.read().split("type = sphere")[1:]:
                c = part.split("vec3(")[1].split(")")[0].split(",")
                r = part.split("radius =")[1].split()[0]
                balls.append([float(np.float32(x)) for x in c + [r]])
        floor = name in ("spheres", "ico5", "ico7", "ico8")
        t = torch.from_numpy(np.concatenate(tris) if tris else np.zeros((0, 9))).cuda()
        _kept[key] = (t, torch.tensor(balls, dtype=torch.float64, device="cuda").reshape(-1, 4), floor)
    return _kept[key]


def _nearest(name, o, d):
    """Closest t of each ray in 64 bits (inf: a miss), and the weights of the
    second and third corner where a triangle is hit, by testing every primitive."""
    tris, balls, floor = _geometry(name)
    n = len(o)
    best = torch.full((n,), math.inf, dtype=torch.float64, device="cuda")
    u = torch.zeros(n, dtype=torch.float64, device="cuda")
    v = torch.zeros(n, dtype=torch.float64, device="cuda")

    def offer(t, a, b, ok):
        nonlocal best, u, v
        ok = ok & (t > 1e-8) & (t < best)
        best, u, v = torch.where(ok, t, best), torch.where(ok, a, u), torch.where(ok, b, v)

    zero = torch.zeros(n, dtype=torch.float64, device="cuda")
    if floor:
        offer(-o[:, 1] / d[:, 1], zero, zero, d[:, 1].abs() > 1e-8)
    for c in balls:
        oc = o - c[:3]
        b = (oc * d).sum(1)
        disc = b * b - ((oc * oc).sum(1) - c[3] * c[3])
        offer(-b - disc.clamp(min=0).sqrt(), zero, zero, disc > 0)
    # with m = o x d, the ray's signed volume against the edge p -> q is
    # d . (p x q) + m . (q - p): six products an edge
    if len(tris):
        ray = torch.cat([d, torch.linalg.cross(o, d)], 1)
        step = max(1, (1 << 27) // n)
        for k in range(0, len(tris), step):
            a, b, c = tris[k:k + step, 0:3], tris[k:k + step, 3:6], tris[k:k + step, 6:9]
            ea, eb, ec = (torch.cat([torch.linalg.cross(p, q), q - p], 1).T.contiguous()
                          for p, q in ((b, c), (c, a), (a, b)))
            nor = torch.linalg.cross(b - a, c - a)
            wa, wb, wc = ray @ ea, ray @ eb, ray @ ec
            inside = ((wa >= 0) & (wb >= 0) & (wc >= 0)) | ((wa <= 0) & (wb <= 0) & (wc <= 0))
            total = wa + wb + wc
            t = ((a * nor).sum(1) - o @ nor.T.contiguous()) / (d @ nor.T.contiguous())
            t = torch.where(inside & (total != 0) & (t > 1e-8), t, math.inf)
            near, at = t.min(1)
            at = at[:, None]
            s = total.gather(1, at)[:, 0]
            offer(near, wb.gather(1, at)[:, 0] / s, wc.gather(1, at)[:, 0] / s, near < math.inf)
    return best, u, v


def exact(case, seed):
    queries = case.get("rays") or case.get("width", 0) * case.get("height", 0)
    if case["kind"] == "serve" or queries * _PRIMS[case["scene"]] > 4e10:
        return None
    if case["kind"] == "trace":
        r0, r1 = _rays(case["scene"], case["rays"], case["how"], seed)
        t, u, v = _nearest(case["scene"], r0[:, :3].double(), r1[:, :3].double())
        return {"t": t, "prim": None, "u": u, "v": v}
    pose = _pose(case["scene"], seed)
    if case.get("integrator", "depth") != "depth" or pose["aperture"] != 0.0:
        return None  # random streams of the package's own, or a value it defines
    # depth: 1 / log(distance) along the pixel centres' rays, the same for every sample
    w, h = case["width"], case["height"]
    pos = torch.tensor(pose["position"], dtype=torch.float64, device="cuda")
    z = torch.tensor(pose["target"], dtype=torch.float64, device="cuda") - pos
    z = z / z.norm()
    x = torch.linalg.cross(torch.tensor([0.0, 1.0, 0.0], dtype=torch.float64, device="cuda"), z)
    x = x / x.norm()
    y = torch.linalg.cross(x, z)
    px = (torch.arange(w, device="cuda", dtype=torch.float64) + 0.5) * 2 / w - 1
    py = ((torch.arange(h, device="cuda", dtype=torch.float64) + 0.5) * 2 / h - 1) * h / w
    d = px[None, :, None] * x + py[:, None, None] * y + z / math.tan(math.radians(pose["fov"]) / 2)
    d = (d / d.norm(dim=2, keepdim=True)).reshape(-1, 3)
    t, _, _ = _nearest(case["scene"], pos.expand(len(d), 3), d)
    v = torch.where(torch.isinf(t), 0.0, 1.0 / torch.log(t.clamp(min=1e-30))).clamp(min=0).reshape(h, w, 1)
    return torch.cat([v, v, v, torch.ones_like(v)], 2)
