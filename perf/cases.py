"""The work users of this framework have it do, as timed cases.

Every case goes through the public entry points (drawlab_amd.Backend and the
C ABI it binds): ray batches against a built scene, the GPU BVH build, whole
renders from a thumbnail to a full-HD frame, shared passes over several
resident scenes, and the learned proposal's training step and guided render.
Scenes and sizes are those of the repository's generators, tests and bench.
"""
import dataclasses
import functools
import math

import numpy as np
import torch

import drawlab_amd
from drawlab_amd import scenes

# Closest-hit and shadow queries per camera path (means over renders of each
# scene at its own depth limits) and a bound on the arithmetic one shading
# vertex cannot do without.
RAYS_PER_PATH = {"cornell_box": (3.7, 1.9), "mis_plates": (2.6, 0.83), "displaced_sphere": (1.97, 0.78),
                 "textured_box": (2.7, 1.3), "material_zoo": (2.3, 1.2), "random": (1.8, 0.32)}
FLOPS_PER_VERTEX = 300
# the network of the learned proposal: 96-64-64-64-64-48
LAYERS = ((96, 64), (64, 64), (64, 64), (64, 64), (64, 48))
PARAMS = sum(i * o + o for i, o in LAYERS)
LOBES = 8


def listed():
    return [
        # a picking or probe query: a thousand rays against a small scene
        {"name": "trace_few", "kind": "trace", "scene": "random", "size": 10_000, "rays": 1_003, "query": "camera"},
        # diffuse-bounce rays of a full-HD frame against the 2M-triangle scene
        {"name": "trace_bounce", "kind": "trace", "scene": "displaced_sphere", "size": 1024, "rays": 4_194_301,
         "query": "bounce"},
        # occlusion queries of a baking pass over a procedural scene
        {"name": "trace_shadow", "kind": "trace", "scene": "random", "size": 500_000, "rays": 1_000_003,
         "query": "shadow"},
        # the acceleration structure of a newly loaded 2M-triangle scene
        {"name": "build_2m", "kind": "build", "scene": "displaced_sphere", "size": 1024, "rays": 65_536},
        # one Adam step of the learned proposal on a batch as renders train it
        {"name": "guide_train", "kind": "guide", "rows": 1 << 18},
        # a thumbnail: the smallest render
        {"name": "render_thumbnail", "kind": "render", "scene": "cornell_box", "size": 0, "width": 64, "height": 64,
         "spp": 4, "mode": "plain"},
        # one frame of a progressive full-HD view of the 2M-triangle scene
        {"name": "render_frame", "kind": "render", "scene": "displaced_sphere", "size": 1024, "width": 1920,
         "height": 1080, "spp": 1, "mode": "progressive"},
        # the Cornell box at its configured size
        {"name": "render_cornell", "kind": "render", "scene": "cornell_box", "size": 0, "width": 512, "height": 512,
         "spp": 64, "mode": "plain"},
        # glossy plates under four lights, an eighth of the configured samples
        {"name": "render_plates", "kind": "render", "scene": "mis_plates", "size": 0, "width": 1280, "height": 720,
         "spp": 64, "mode": "plain"},
        # the 2M-triangle scene under the sky, one default pass at full HD
        {"name": "render_sphere", "kind": "render", "scene": "displaced_sphere", "size": 1024, "width": 1920,
         "height": 1080, "spp": 64, "mode": "plain"},
        # what the render service runs: images of several resident scenes
        # (every BSDF, textures, point and area lights) in one pass
        {"name": "batch_scenes", "kind": "batch", "images": 9, "width": 333, "height": 251, "spp": 16},
        # directions from the learned proposal, its network not trained on
        {"name": "render_guided", "kind": "render", "scene": "displaced_sphere", "size": 256, "width": 480,
         "height": 270, "spp": 64, "mode": "guided"},
    ]


def _log(rng, lo, hi):
    """An integer between lo and hi, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "trace", "build", "guide", "render", "render", "render", "batch"])
    if kind == "guide":
        return {"kind": "guide", "rows": _log(rng, 1_000, 1 << 18)}
    if kind == "batch":
        images = rng.randint(2, 16)
        width = _log(rng, 48, 512)
        height = max(32, int(width * rng.uniform(0.5, 1.2)))
        spp = max(1, min(_log(rng, 1, 64), 30_000_000 // (images * width * height)))
        return {"kind": "batch", "images": images, "width": width, "height": height, "spp": spp}
    scene = rng.choice(["random", "displaced_sphere"] + (["cornell_box", "mis_plates", "textured_box", "material_zoo"]
                                                         if kind == "render" else []))
    size = {"random": _log(rng, 5_000, 500_000), "displaced_sphere": _log(rng, 24, 1024)}.get(scene, 0)
    if kind == "trace":
        return {"kind": "trace", "scene": scene, "size": size, "rays": _log(rng, 700, 4_100_000),
                "query": rng.choice(["camera", "bounce", "shadow"])}
    if kind == "build":
        return {"kind": "build", "scene": scene, "size": size, "rays": 65_536}
    width = _log(rng, 48, 1920)
    height = max(32, min(1080, int(width * rng.uniform(0.5, 1.0))))
    mode = rng.choice(["plain", "plain", "plain", "progressive", "guided"])
    most = {"plain": 60_000_000, "progressive": 4 * width * height, "guided": 8_000_000}[mode]
    spp = max(1, min(_log(rng, 1, 256), most // (width * height)))
    return {"kind": "render", "scene": scene, "size": size, "width": width, "height": height, "spp": spp, "mode": mode}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=8)
def _scene(name, size):
    if name == "displaced_sphere":
        level = max(1, min(5, int(math.log(max(size, 2), 4))))
        return scenes.displaced_sphere(grid=size, glass_level=level)
    if name == "random":
        return scenes.random_scene(102, size)
    return getattr(scenes, name)()


def _desc(name, size, width, height, seed):
    """The scene seen by a camera of this size whose eye the seed moves a little."""
    d = _scene(name, size)
    r = np.random.default_rng(seed)
    span = float(np.linalg.norm(np.subtract(d.camera.lookat, d.camera.eye)))
    eye = tuple(float(e + 0.02 * span * r.uniform(-1, 1)) for e in d.camera.eye)
    return dataclasses.replace(d, camera=dataclasses.replace(d.camera, eye=eye, width=width, height=height))


def _loaded(desc):
    be = drawlab_amd.Backend(0)
    be.upload_scene(desc)
    be.build_accel(drawlab_amd.BUILD_GPU)
    return be


def _camera_rays(desc, g):
    """One ray per pixel, rows in order, through a jittered film position."""
    cd = drawlab_amd.camera_desc(desc.camera)
    w, h = desc.camera.width, desc.camera.height
    eye, U, V, W = (torch.tensor(list(getattr(cd, k)), device="cuda") for k in ("eye", "U", "V", "W"))
    y, x = torch.meshgrid(torch.arange(h, device="cuda"), torch.arange(w, device="cuda"), indexing="ij")
    j = torch.rand((2, h, w), generator=g, device="cuda")
    dx = (x + j[0]) / w * 2 - 1
    dy = (h - y - j[1] - 1) / h * 2 - 1
    d = (dx[..., None] * U + dy[..., None] * V + W).reshape(-1, 3)
    return eye.expand(w * h, 3), torch.nn.functional.normalize(d, dim=1)


def _planes(o, d, tmin, tmax):
    """Rays as the trace entry points take them: 8 planes of n floats."""
    n = o.shape[0]
    return torch.cat([o.T, d.T, torch.full((1, n), tmin, device="cuda"),
                      torch.full((1, n), tmax, device="cuda")]).contiguous().float()


def _trace(be, rays, out):
    n = rays.shape[1]
    be._check(be.L.dl_hip_trace_closest(be.h, rays.data_ptr(), n, *(out[k].data_ptr() for k in ("prim", "t", "u", "v"))))


def _hits(n):
    return {"prim": torch.empty(n, dtype=torch.int32, device="cuda"),
            **{k: torch.empty(n, device="cuda") for k in ("t", "u", "v")}}


def _vertices(desc):
    """(triangles, 3, 3) vertex positions in global primitive order."""
    return torch.cat([torch.from_numpy(np.ascontiguousarray(m.V[m.F.astype(np.int64)])).cuda() for m in desc.meshes])


def _batch_rays(be, desc, query, n, seed):
    """n rays: camera rays row by row, or rays leaving the points that camera
    rays hit, in their order -- cosine-distributed about the face normal (as
    diffuse bounces leave) or toward the scene's sky and lamps (as emitter
    samples do)."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    if query == "camera":
        return _planes(*_camera_rays(desc, g), 1e-4, math.inf)[:, :n].contiguous()
    o, d = _camera_rays(desc, g)
    rays, out = _planes(o, d, 1e-4, math.inf), _hits(o.shape[0])
    torch.cuda.synchronize()
    _trace(be, rays, out)
    seen = torch.nonzero(out["prim"] >= 0)[:, 0]
    pick = seen[(torch.arange(n, device="cuda") * seen.numel()) // n]
    tri = _vertices(desc)[out["prim"][pick].long()]
    u, v = out["u"][pick, None], out["v"][pick, None]
    p = tri[:, 0] * (1 - u - v) + tri[:, 1] * u + tri[:, 2] * v
    nrm = torch.nn.functional.normalize(torch.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0], dim=1), dim=1)
    nrm = torch.where((nrm * d[pick]).sum(1, keepdim=True) > 0, -nrm, nrm)
    ball = torch.nn.functional.normalize(torch.randn((n, 3), generator=g, device="cuda"), dim=1)
    cosine = torch.nn.functional.normalize(nrm + 0.999 * ball, dim=1)
    if query == "bounce":
        return _planes(p, cosine, 1e-4, math.inf)
    # three emitter samples in four go to a small bright region
    lamp = torch.tensor([0.5, 0.7071, 0.5], device="cuda") + 0.02 * ball
    lamp = torch.nn.functional.normalize(lamp, dim=1)
    use = (torch.rand((n, 1), generator=g, device="cuda") < 0.75) & ((lamp * nrm).sum(1, keepdim=True) > 0)
    return _planes(p, torch.where(use, lamp, cosine), 1e-4, 1e16)


def _train_batch(rows, seed):
    """Network inputs of `rows` shading points (positions on a few surfaces,
    encoded as the network takes them), directions toward a few bright
    regions, and training weights of a heavy-tailed distribution."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    pos = torch.rand((rows, 3), generator=g, device="cuda")
    wall = torch.randint(0, 3, (rows,), generator=g, device="cuda")
    pos[torch.arange(rows, device="cuda"), wall] = (torch.rand(rows, generator=g, device="cuda") < 0.5).float()
    angle = pos[:, :, None] * (math.pi * 2.0 ** torch.arange(12, device="cuda"))
    x = torch.zeros((rows, 96), device="cuda")
    x[:, :72] = torch.stack([angle.sin(), angle.cos()], -1).reshape(rows, 72)

    def unit():
        return torch.nn.functional.normalize(torch.randn((rows, 3), generator=g, device="cuda"), dim=1)

    x[:, 72:75], x[:, 75:78] = unit(), unit()
    x[:, 78] = torch.where(torch.rand(rows, generator=g, device="cuda") < 0.7, 1.0, 0.4)
    lamps = torch.nn.functional.normalize(torch.randn((4, 3), generator=g, device="cuda"), dim=1)
    at = lamps[torch.randint(0, 4, (rows,), generator=g, device="cuda")] + 0.3 * unit()
    w = torch.rand(rows, generator=g, device="cuda").pow(4)
    return x, torch.nn.functional.normalize(at, dim=1).contiguous(), w


BATCH_SCENES = (("cornell_box", 0), ("textured_box", 0), ("material_zoo", 0), ("random", 50_000))


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": dict(case), "seed": int(seed)}
    if kind == "guide":
        be = drawlab_amd.Backend(0)
        be.guide_init(seed=seed, lr=1e-2)
        x, d, w = _train_batch(case["rows"], seed)
        state.update(be=be, x=x, d=d, w=w)
    elif kind == "batch":
        be = drawlab_amd.Backend(0)
        items = []
        for k, (name, size) in enumerate(BATCH_SCENES[:case["images"]]):
            be.upload_scene(_desc(name, size, 64, 64, seed))
            be.build_accel(drawlab_amd.BUILD_GPU)
            be.scene_keep(k + 1)
        for i in range(case["images"]):
            name, size = BATCH_SCENES[i % len(BATCH_SCENES)]
            cam = _desc(name, size, case["width"] + 8 * i, case["height"], seed + i).camera
            items.append({"camera": cam, "spp": case["spp"], "seed": seed + i, "film": i,
                          "scene": 1 + i % len(BATCH_SCENES)})
        state.update(be=be, items=items)
    elif kind in ("trace", "build"):
        side = max(8, int(math.ceil(math.sqrt(min(case["rays"], 1 << 21)))))
        if case.get("query") == "camera":
            side = int(math.ceil(math.sqrt(case["rays"])))
        desc = _desc(case["scene"], case["size"], side, side, seed)
        be = _loaded(desc)
        state.update(be=be, desc=desc, rays=_batch_rays(be, desc, case.get("query", "camera"), case["rays"], seed))
        n = state["rays"].shape[1]
        state["out"] = ({"occluded": torch.empty(n, dtype=torch.uint8, device="cuda")}
                        if case.get("query") == "shadow" else _hits(n))
    else:
        be = _loaded(_desc(case["scene"], case["size"], case["width"], case["height"], seed))
        if case["mode"] == "guided":
            be.guide_init(seed=seed)
        state.update(be=be, frame=0)
    torch.cuda.synchronize()
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case, be = state["case"], state["be"]
    kind = case["kind"]
    if kind == "trace":
        if case["query"] == "shadow":
            be._check(be.L.dl_hip_trace_shadow(be.h, state["rays"].data_ptr(), state["rays"].shape[1],
                                               state["out"]["occluded"].data_ptr()))
        else:
            _trace(be, state["rays"], state["out"])
        return state["out"]
    if kind == "build":
        # the structure itself is read by the queries that follow it
        be.build_accel(drawlab_amd.BUILD_GPU)
        _trace(be, state["rays"], state["out"])
        return state["out"]
    if kind == "guide":
        loss = drawlab_amd.ctypes.c_float()
        be._check(be.L.dl_hip_guide_train_step(be.h, state["x"].data_ptr(), state["d"].data_ptr(),
                                               state["w"].data_ptr(), case["rows"], 1,
                                               drawlab_amd.ctypes.byref(loss)))
        return {"loss": float(loss.value), "params": be.guide_params()[0]}
    if kind == "batch":
        images, st = be.render_batch(state["items"])
        return {"images": images, "closest": st["closest_rays"], "shadow": st["shadow_rays"]}
    progressive = case["mode"] == "progressive"
    guided = case["mode"] == "guided"
    image, st = be.render(spp=case["spp"], seed=state["seed"], first_sample=state["frame"] if progressive else 0,
                          accumulate=progressive, guided=guided, guide_frozen=guided)
    state["frame"] += case["spp"]
    return {"image": image, "closest": st["closest_rays"], "shadow": st["shadow_rays"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far results may lie apart
# ---------------------------------------------------------------------------
def _triangles(name, size):
    return _scene(name, size).num_triangles


def _ray_flops(tris):
    """Four box tests per level of a four-way tree and two triangle tests."""
    return 4 * 24 * max(1.0, math.log(tris, 4)) + 2 * 52


def work(case):
    kind = case["kind"]
    if kind == "guide":
        n = case["rows"]
        # inputs once; forward, and the two products of the backward pass
        return {"bytes": n * 4 * (96 + 3 + 1) + 2 * 4 * PARAMS,
                "flops": n * (2 * 3 * sum(i * o for i, o in LAYERS) - 2 * 96 * 64)}
    if kind == "batch":
        paths = sum((case["width"] + 8 * i) * case["height"] for i in range(case["images"])) * case["spp"]
        return {"bytes": 12 * paths // case["spp"] + 112 * 55_000,
                "flops": paths * (3.6 * _ray_flops(10_000) + 2.5 * FLOPS_PER_VERTEX)}
    tris = _triangles(case["scene"], case["size"])
    if kind == "trace":
        out = 1 if case["query"] == "shadow" else 16
        return {"bytes": case["rays"] * (32 + out) + 76 * tris, "flops": case["rays"] * _ray_flops(tris)}
    if kind == "build":
        # vertices and indices in; triangles of 48 bytes and nodes out
        return {"bytes": tris * (18 + 12 + 48 + 28) + case["rays"] * 48, "flops": case["rays"] * _ray_flops(tris)}
    paths = case["width"] * case["height"] * case["spp"]
    closest, shadow = RAYS_PER_PATH[case["scene"]]
    return {"bytes": 12 * case["width"] * case["height"] + 112 * tris,
            "flops": paths * ((closest + shadow) * _ray_flops(tris) + closest * FLOPS_PER_VERTEX)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("trace", "build"):
        # the nearest (t, primitive) over all triangles is one answer,
        # whatever tree and order it is found in
        return "exact"
    if kind == "guide":
        # rows summed in another order move the parameters by 3e-6 at most;
        # a first Adam step moves a weight by the rate times the gradient's
        # sign, so one weight whose gradient is nearly zero may differ by
        # twice that: 1e-3 of the parameters' norm
        return {"rel": 1e-3, "max": 0.3}
    if case.get("mode") == "guided":
        # another rounding of a bfloat16 weight or activation moves sampled
        # directions and with them, now and then, a whole path: parameters
        # scaled by 1 + 1e-6 give images 2e-3 apart (0.11 at one pixel)
        return {"rel": 8e-3, "max": 0.43}
    # per-path arithmetic is pinned bit for bit; the film's sums are 32 bits
    return {"rel": 1e-5, "max": 1e-3}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _exact_hits(rays, tri):
    """Nearest hits of every ray by testing every triangle."""
    o, d = rays[0:3].T.double(), rays[3:6].T.double()
    tri = tri.double()
    e1, e2 = tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    best = [torch.empty(o.shape[0], dtype=torch.float64, device="cuda") for _ in range(3)]
    for s in range(0, o.shape[0], 64):
        oo, dd = o[s:s + 64, None], d[s:s + 64, None]
        p = torch.cross(dd.expand(-1, tri.shape[0], -1), e2[None].expand(dd.shape[0], -1, -1), dim=2)
        det = (e1 * p).sum(2)
        tv = oo - tri[None, :, 0]
        u = (tv * p).sum(2) / det
        q = torch.cross(tv, e1[None].expand(dd.shape[0], -1, -1), dim=2)
        v = (dd * q).sum(2) / det
        t = (e2 * q).sum(2) / det
        ok = (det.abs() >= 1e-8) & (u >= 0) & (u <= 1) & (v >= 0) & (u + v <= 1)
        ok &= (t >= rays[6, s:s + 64, None]) & (t <= rays[7, s:s + 64, None])
        t = torch.where(ok, t, math.inf)
        m, k = t.min(1)
        miss = torch.isinf(m)
        best[0][s:s + 64] = torch.where(miss, rays[7, s:s + 64].double(), m)
        for b, a in ((best[1], u), (best[2], v)):
            b[s:s + 64] = torch.where(miss, 0.0, a.gather(1, k[:, None])[:, 0])
    return {"prim": None, "t": best[0], "u": best[1], "v": best[2]}


def _bf16(a):
    return a.float().bfloat16().double()


def _exact_step(theta, x, d, w, lr):
    """One training step in float64; the network's weights, activations and
    the gradients its matrix products read are bfloat16 by definition."""
    W, b, o = [], [], 0
    for i, k in LAYERS:
        W.append(theta[o:o + i * k].reshape(k, i))
        b.append(theta[o + i * k:o + i * k + k])
        o += i * k + k
    acts = [_bf16(x)]
    for l in range(4):
        acts.append(_bf16(torch.relu(acts[l] @ _bf16(W[l]).T + b[l])))
    out = (acts[4] @ _bf16(W[4]).T + b[4]).detach().requires_grad_(True)
    lobe = out[:, :5 * LOBES].reshape(-1, LOBES, 5)
    kappa = torch.exp(-3.0 + 10.0 * torch.sigmoid(lobe[..., 1]))
    mu = lobe[..., 2:] / lobe[..., 2:].norm(dim=2, keepdim=True).clamp_min(1e-6)
    logf = torch.log(kappa / (2 * math.pi * -torch.expm1(-2 * kappa))) + kappa * ((mu * d.double()[:, None]).sum(2) - 1)
    logq = torch.logsumexp(torch.log_softmax(lobe[..., 0], 1) + logf, 1)
    c = w.double()
    loss = -(c * logq.clamp_min(math.log(1e-30))).sum() / c.sum()
    loss.backward()
    g, grads = out.grad, [None] * 5
    for l in range(4, -1, -1):
        grads[l] = torch.cat([(_bf16(g).T @ acts[l]).reshape(-1), g.sum(0)])
        if l:
            g = (_bf16(g) @ _bf16(W[l])) * (acts[l] > 0)
    grad = torch.cat(grads)
    return float(loss), theta - lr * grad / (grad.abs() + 1e-8)


def exact(case, seed):
    if case["kind"] == "guide":
        s = prepare(case, seed)
        theta = torch.from_numpy(s["be"].guide_params()[0]).cuda().double()
        loss, params = _exact_step(theta, s["x"], s["d"], s["w"], 1e-2)
        return {"loss": loss, "params": params.cpu().numpy()}
    if case["kind"] == "trace" and case["query"] != "shadow":
        tris = _triangles(case["scene"], case["size"])
        if case["rays"] * tris > 2e9:
            return None
        s = prepare(case, seed)
        return _exact_hits(s["rays"], _vertices(s["desc"]))
    return None
