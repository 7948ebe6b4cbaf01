"""The work that programs using this renderer have it do, as measurable cases.

A case is a dict of plain values:

  kind      "frame"     render_frame: a scene the renderer has not seen (upload,
                        BVH build, every sample, RGBA8 image): the CLI, a thumbnailer
            "resident"  restart_frame + one pass of every sample: a still or an
                        animation frame re-rendered with the scene on the GPU
            "editor"    restart_frame + render_sample once per sample: the
                        viewport refining after a change
            "drag"      new_frame + one render_sample: the viewport while an
                        object is dragged (a new scene for every image)
            "noalloc"   rd_render_frame_noalloc
            "batch"     BatchRenderer.render of `jobs` scenes at once
  scene     "small" (9 objects), "plain" (97 spheres and cubes), "clustered"
            (`objects` of them), "room" (`objects` inside a closed diffuse
            sphere, lamps, no sky: every path runs to the bounce limit),
            "benchmark" (raydar's own scene file, 183 objects)
  width, height, spp, bounces
  vulkan    True: the Vulkan renderer's semantics
  hdr       True: the program reads the float accumulator too

Seeds make both the scene (but for the scene file) and the random numbers.
"""
import ctypes
import math
import os

import numpy as np
import torch

import raydar_amd as ra
from raydar_amd import abi, scenegen
from raydar_amd.batch import BatchRenderer, Job
from raydar_amd.scene import Scene, make_object, solid_world

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _case(kind, scene, width, height, spp, bounces=12, objects=0, vulkan=False, hdr=False):
    return dict(kind=kind, scene=scene, objects=objects, width=width, height=height, spp=spp,
                bounces=bounces, vulkan=vulkan, hdr=hdr)


def listed():
    cases = [
        # a thumbnail in a scene browser: the smallest whole call
        ("thumbnail_128", _case("frame", "clustered", 128, 128, 8, 4, objects=64, hdr=True)),
        # a preview of a small scene, scene upload and BVH build included
        ("preview_256", _case("frame", "small", 256, 256, 16, hdr=True)),
        # an object dragged in the viewport at full HD: one sample per change
        ("drag_1080p", _case("drag", "plain", 1920, 1080, 1)),
        # the viewport refining at full HD, an image after every sample
        ("editor_1080p", _case("editor", "plain", 1920, 1080, 8)),
        # a frame of no round size, few samples, a mid-size scene
        ("odd_643x361", _case("frame", "clustered", 643, 361, 7, 8, objects=300, hdr=True)),
        # an interior: no sky, every path runs to the bounce limit
        ("room_540p", _case("resident", "room", 960, 540, 16, objects=40, hdr=True)),
        # a still of the usual size and quality (the headline workload)
        ("plain_1080p", _case("resident", "plain", 1920, 1080, 64)),
        # the same in a scene of 4096 objects, whose tree does not fit a CU's LDS
        ("clustered_1080p", _case("resident", "clustered", 1920, 1080, 64, objects=4096)),
        # raydar's benchmark scene at its own 4K resolution
        ("benchmark_4k", _case("frame", "benchmark", 3840, 2160, 8)),
        # the Vulkan renderer's images
        ("vulkan_720p", _case("resident", "plain", 1280, 720, 16, vulkan=True)),
        # a render inside a program that cannot allocate device memory
        ("noalloc_720p", _case("noalloc", "plain", 1280, 720, 8)),
        # a farm's batch: 16 scenes of 16-2048 objects, 128^2 to 1024x768
        ("batch_16", dict(kind="batch", jobs=16, scene="clustered", max_width=1024)),
    ]
    return [dict(c, name=n) for n, c in cases]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "resident", "resident", "editor", "drag", "noalloc", "vulkan",
                       "batch"])
    if kind == "batch":
        return dict(kind="batch", jobs=rng.randint(3, 20), scene="clustered",
                    max_width=rng.choice([256, 512, 1024]))
    vulkan = kind == "vulkan"
    kind = "resident" if vulkan else kind
    width = _log(rng, 64, 2560)
    height = max(48, min(1440, int(width * rng.uniform(0.45, 1.1))))
    scene = rng.choice(["small", "plain", "plain", "clustered", "clustered", "room"])
    spp = {"drag": 1, "editor": rng.randint(2, 12)}.get(kind) or _log(rng, 1, 96)
    # nothing dearer than the 1080p still (the Vulkan images cost more each path, the
    # allocation-free call renders in short passes)
    most = {"noalloc": 12e6, "editor": 24e6}.get(kind, 16e6 if vulkan else 60e6)
    if scene == "room":
        most /= 4
    spp = max(1, min(spp, int(most / (width * height))))
    if kind == "noalloc" and width * height > 1920 * 1080:
        width, height = 1920, 1080
    objects = {"clustered": _log(rng, 5, 4096), "room": _log(rng, 4, 200)}.get(scene, 0)
    return _case(kind, scene, width, height, spp, rng.choice([4, 8, 12, 12, 16]), objects, vulkan,
                 hdr=rng.random() < 0.3)


# ------------------------------------------------------------- scenes ------
def _room(seed, objects, width, height):
    rng = scenegen.SplitMix64(seed ^ 0x600D)
    objs = [make_object(abi.RD_SPHERE, (0.0, 5.0, 0.0), 16.0, albedo=(0.75, 0.75, 0.7), roughness=1.0)]
    for i in range(objects):
        size = rng.uniform(0.3, 1.5)
        centre = (rng.uniform(-7, 7), rng.uniform(-3, 9), rng.uniform(-8, 4))
        m = scenegen.material(rng, rng.choice(4))
        if i % 8 == 0:
            m.update(emission_color=(1.0, 0.9, 0.7), emission_strength=rng.uniform(2.0, 12.0))
        objs.append(make_object(abi.RD_CUBE if i % 3 == 2 else abi.RD_SPHERE, centre, size, **m))
    return Scene(scenegen.small_camera(width, height), solid_world((0.0, 0.0, 0.0)), np.array(objs))


def _scene(case, seed):
    w, h = case["width"], case["height"]
    if case["scene"] == "small":
        s = scenegen.plain_small(seed)
        return Scene(scenegen.small_camera(w, h), s.world, s.objects)
    if case["scene"] == "plain":
        return scenegen.plain_1080p(seed, w, h)
    if case["scene"] == "room":
        return _room(seed, case["objects"], w, h)
    if case["scene"] == "benchmark":
        return Scene.load(os.path.join(ROOT, "tests", "golden", "benchmark.rscn"))
    return scenegen.clustered(seed, case["objects"], w, h)


def _batch_specs(case, seed):
    """Jobs of the shapes scenegen.batch_jobs draws; `seed` makes the scenes."""
    sizes = [r for r in scenegen.RESOLUTIONS_BATCH if r[0] <= case["max_width"]]
    specs = []
    for i in range(case["jobs"]):
        rng = scenegen.SplitMix64((1000 + i) ^ 0xB47C4)
        n = int(round(rng.log_uniform(16, 2048)))
        w, h = sizes[rng.choice(len(sizes))]
        spp, bounces = (8, 32)[rng.choice(2)], (4, 8, 12)[rng.choice(3)]
        s = 64 * seed + i
        specs.append(scenegen.Job(scenegen.clustered(s, n, w, h), spp, bounces, s))
    return specs


# -------------------------------------------------------------- the pass ---
def prepare(case, seed):
    if case["kind"] == "batch":
        jobs = [Job(j.scene, j.spp, j.bounces, j.seed) for j in _batch_specs(case, seed)]
        return dict(case=case, renderer=BatchRenderer(), jobs=jobs)
    sc = _scene(case, seed)
    r = ra.HipRenderer(max_sample_count=case["spp"], max_bounces=case["bounces"], seed=seed,
                       semantics=1 if case["vulkan"] else 0)
    state = dict(case=case, renderer=r, scene=sc, out=np.zeros((sc.height, sc.width, 4), np.uint8))
    if case["kind"] == "resident":
        r.set_samples_per_pass(case["spp"])
    if case["kind"] in ("resident", "editor"):
        r.new_frame(sc)
    if case["kind"] == "noalloc":
        f = ra.lib().rd_render_frame_noalloc
        f.restype = ctypes.c_int
        f.argtypes = [ctypes.c_void_p, ctypes.POINTER(abi.RdScene), ctypes.c_void_p, ctypes.c_size_t]
        state["rd_scene"] = sc.as_rd()
    return state


def run(state):
    case, r = state["case"], state["renderer"]
    kind = case["kind"]
    if kind == "batch":
        r.render(state["jobs"])
        return [[j.rgba, j.acc] for j in state["jobs"]]
    out = state["out"]
    if kind == "frame":
        r.render_frame(state["scene"], out)
    elif kind == "drag":
        r.new_frame(state["scene"])
        r.render_sample(out=out)
    elif kind == "noalloc":
        ra.check(ra.lib().rd_render_frame_noalloc(r._h, ctypes.byref(state["rd_scene"]),
                                                  out.ctypes.data_as(ctypes.c_void_p), out.nbytes), r._h)
    else:
        r.restart_frame()
        for _ in range(case["spp"] if kind == "editor" else 1):
            r.render_sample(out=out)
    # (the allocation-free call keeps no accumulator a program could read)
    return [out, r.accumulator()] if case["hdr"] and kind != "noalloc" else [out]


def _sizes(case):
    """(pixels, samples, bounces, objects) of each image."""
    if case["kind"] == "batch":
        return [(j.scene.width * j.scene.height, j.spp, j.bounces, len(j.scene.objects))
                for j in _batch_specs(case, 1)]
    n = {"small": 9, "plain": 97, "benchmark": 183, "room": case["objects"] + 1}
    return [(case["width"] * case["height"], case["spp"], case["bounces"],
             n.get(case["scene"], case["objects"]))]


def work(case):
    """Bytes: each scene's objects (64 B) and tree read once, its images written
    once.  FP32 operations: a path of this renderer's scenes takes about 300
    plus 100 for each bounce it may make, in box and primitive tests through a
    tree, shading and the camera ray (counted on the 97- and the 4096-object
    scene: about 1500 at 12 bounces); in a closed room, where every path
    runs to the limit, three times as many."""
    nbytes = flops = 0
    for px, spp, bounces, objects in _sizes(case):
        images = case["spp"] if case["kind"] == "editor" else 1
        hdr = case["kind"] == "batch" or (case["hdr"] and case["kind"] != "noalloc")
        nbytes += 192 * objects + px * (4 * images + (16 if hdr else 0))
        flops += px * spp * (300 + 100 * bounces) * (3 if case["scene"] == "room" else 1)
    return {"bytes": nbytes, "flops": flops}


# ------------------------------------------------------------- in 64 bits --
# The CPU renderer's paths in float64 torch, every object tested against every
# ray.  A path is a chain of decisions (which object, which branch), so this
# value and a 32-bit image part where a decision falls differently.
def exact(case, seed):
    if case["kind"] == "batch" or case["vulkan"] or not case["hdr"] or case["kind"] == "noalloc":
        return None
    sc = _scene(case, seed)
    if sc.width * sc.height * case["spp"] * len(sc.objects) > 1.2e9:
        return None
    if case["scene"] == "room":
        return None  # paths this long part too often for the two to be compared
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    npix = sc.width * sc.height
    acc = torch.zeros((npix, 4), dtype=torch.float64, device=dev)
    for sample in range(case["spp"]):
        acc[:, :3] += _sample64(sc, sample, case["bounces"], seed, dev)
        acc[:, 3] += 1.0
    return [None, acc.cpu().numpy()]


def _philox(c, key):
    """Philox-4x32-10 over int64 tensors holding 32-bit words."""
    mask = 0xFFFFFFFF
    c0, c1, c2, c3 = c
    k0, k1 = key & mask, key >> 32
    for i in range(10):
        if i:
            k0, k1 = (k0 + 0x9E3779B9) & mask, (k1 + 0xBB67AE85) & mask
        p0, p1 = 0xD2511F53 * c0, 0xCD9E8D57 * c2
        c0, c1, c2, c3 = (((p1 >> 32) & mask) ^ c1 ^ k0, p1 & mask,
                          ((p0 >> 32) & mask) ^ c3 ^ k1, p0 & mask)
    return [(w >> 8).double() * 2.0 ** -24 for w in (c0, c1, c2, c3)]


def _dot(a, b):
    return (a * b).sum(-1)


def _unit(v):
    return v / _dot(v, v).sqrt()[:, None]


def _trace64(objs, o, d):
    """Nearest hit: (distance, object index or -1); the first of equal distances."""
    best = torch.full_like(o[:, 0], math.inf)
    idx = torch.full_like(best, -1, dtype=torch.int64)
    a = _dot(d, d)
    for i, ob in enumerate(objs):
        c = torch.tensor(ob["center"].astype(np.float64), device=o.device)
        size = float(ob["size"])
        if ob["kind"] == abi.RD_SPHERE:
            oc = o - c
            k = _dot(oc, d)
            disc = k * k - a * (_dot(oc, oc) - size * size)
            s = disc.clamp(min=0.0).sqrt()
            t = torch.where(-k - s >= 0, (-k - s) / a, (-k + s) / a)
            hit = (disc >= 0) & (t >= 0)
        else:
            t1, t2 = (c - size / 2 - o) / d, (c + size / 2 - o) / d
            near = torch.minimum(t1, t2).amax(-1)
            far = torch.maximum(t1, t2).amin(-1)
            t = torch.where(near < 0, far, near)
            hit = (far >= 0) & (near <= far)
        better = hit & (t < best)
        best = torch.where(better, t, best)
        idx = torch.where(better, torch.full_like(idx, i), idx)
    return best, idx


def _sky64(world, d):
    if world["kind"] == abi.RD_WORLD_SOLID_COLOR:
        return torch.tensor(world["solid_color"], dtype=torch.float64, device=d.device).expand_as(d)
    lo, hi = (torch.tensor(world[k], dtype=torch.float64, device=d.device)
              for k in ("bottom_color", "top_color"))
    return lo + (hi - lo) * ((_unit(d)[:, 1] + 1.0) * 0.5)[:, None]


def _sample64(sc, sample, bounces, seed, dev):
    W, H = sc.width, sc.height
    n = W * H
    cam = sc.camera

    def mat(k):
        return torch.tensor(cam[k], dtype=torch.float64, device=dev).reshape(4, 4)  # rows are columns

    px = torch.arange(n, device=dev)
    uv = torch.stack([(px % W).double() / W * 2 - 1, (1 - (px // W).double() / H) * 2 - 1,
                      -torch.ones(n, dtype=torch.float64, device=dev),
                      -torch.ones(n, dtype=torch.float64, device=dev)], 1)
    p = uv @ mat("inverse_proj_matrix")
    d = -_unit(((p / p[:, 3:]) @ mat("inverse_view_matrix"))[:, :3])
    o = torch.tensor(cam["position"], dtype=torch.float64, device=dev).expand(n, 3)
    ob = sc.objects

    def col(k):
        return torch.tensor(ob[k].astype(np.float64), device=dev)

    f = {k: col(k) for k in ("center", "size", "albedo", "roughness", "metallic", "transmission", "ior")}
    emission = col("emission_color") * col("emission_strength")[:, None]
    cube = torch.tensor(ob["kind"] == abi.RD_CUBE, device=dev)
    out = torch.zeros((n, 3), dtype=torch.float64, device=dev)
    light, att = torch.zeros_like(out), torch.ones_like(out)
    zero = torch.zeros_like(px)
    for bounce in range(bounces):
        t, i = _trace64(ob, o, d)
        miss = i < 0
        out[px[miss]] = light[miss] + _sky64(sc.world, d[miss]) * att[miss]
        px, o, d, t, i, light, att = (v[~miss] for v in (px, o, d, t, i, light, att))
        if len(px) == 0:
            return out
        pos = o + d * t[:, None]
        l = pos - f["center"][i]
        far = (l.abs() - f["size"][i][:, None] / 2).abs()
        axis = torch.where((far[:, 0] < far[:, 1]) & (far[:, 0] < far[:, 2]), 0,
                           torch.where(far[:, 1] < far[:, 2], 1, 2))
        face = torch.zeros_like(l).scatter_(1, axis[:, None], torch.copysign(
            torch.ones_like(t), l.gather(1, axis[:, None])[:, 0])[:, None])
        nrm = torch.where(cube[i][:, None], face, _unit(l))
        front = _dot(nrm, d) <= 0
        nrm = torch.where(front[:, None], nrm, -nrm)
        z = zero[:len(px)]
        u = [_philox((px, z + sample, z + (4 * bounce + b), z), seed) for b in (0, 1)]
        rnd = _unit(torch.stack(u[1][:3], 1) * 2 - 1)
        rough = f["roughness"][i] ** 2
        diffuse = nrm + rnd
        diffuse = torch.where((_dot(diffuse, nrm) < 0)[:, None], -diffuse, diffuse)
        mirror = d - 2 * _dot(d, nrm)[:, None] * nrm
        glass = u[0][0] < f["transmission"][i]
        eta = torch.where(front, 1 / f["ior"][i], f["ior"][i])
        du = _unit(d)
        cos = (-_dot(du, nrm)).clamp(max=1.0)
        r0 = ((eta - 1) / (eta + 1)) ** 2
        fresnel = r0 + (1 - r0) * (1 - cos) ** 5
        bends = glass & (fresnel < u[0][1]) & (eta * (1 - cos * cos).clamp(min=0).sqrt() <= 1)
        perp = (du + nrm * cos[:, None]) * eta[:, None]
        refracted = perp - nrm * (1 - _dot(perp, perp)).abs().sqrt()[:, None]
        bent = _unit(torch.where(bends[:, None], refracted, mirror) + rnd * rough[:, None])
        scatters = ~glass & ~(u[0][1] < f["metallic"][i]) & (u[0][2] < rough)
        d = torch.where(scatters[:, None], diffuse, bent)
        o = pos + torch.where(glass[:, None], d, nrm) * 1e-4
        d = torch.where((_dot(d, d) < 1e-10)[:, None], nrm, d)
        light, att = light + emission[i], att * f["albedo"][i]
    out[px] = light
    return out
