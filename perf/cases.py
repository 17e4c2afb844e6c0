"""Timed workloads: what programs that use this package have it do.

A program builds or loads an octree on the host, uploads it once
(DeviceTree), and then, again and again: renders viewports, casts its own ray
sets (picking, line of sight, secondary rays), draws shaded images, does the
same at a level of detail, hands many views over many trees to one batched
run, and edits the tree and looks again. One case is one such call, with the
package's default settings.

Scenes are the package's own seeded ones (caves, heightfields, spheres) and a
small landscape inserted voxel by voxel. The 2048^3 spheres of the full
benchmark are left out: building them takes minutes of host time; the
heightfield of 1024^3 and the spheres of 512^3 with their brick dimension
stand for large trees here.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from shocovox_amd import Batch, DeviceTree, Octree, Viewport, alloc_hits

SCENES = {"caves": 2, "spheres": 3, "heights": 4}
FIELDS = {
    # everything a hit carries (the default of render() and cast())
    "all": ("hit", "pix", "albedo", "voxel", "distance", "impact", "normal", "flags"),
    # what a viewer needs: 24 bytes a ray
    "view": ("hit", "albedo", "voxel", "distance"),
}
BYTES = {"hit": 4, "pix": 4, "albedo": 4, "voxel": 12, "distance": 4, "impact": 12, "normal": 12,
         "flags": 4}
# a ray's own arithmetic (setup, 11 DDA steps, the hit): about what the caves
# need on average
FLOPS_PER_RAY = 230
RESOLUTIONS = ((128, 128), (512, 512), (1280, 720))


def listed():
    return [
        # line-of-sight queries of a game step: a handful of rays, one answer
        # each; latency and the launch are everything
        {"name": "pick_1k", "kind": "cast", "scene": "hills", "size": 64, "dim": 8, "rays": 1009,
         "fields": "all"},
        # a thumbnail of a small tree
        {"name": "frame_256", "kind": "frame", "scene": "hills", "size": 64, "dim": 4,
         "width": 256, "height": 256, "fields": "all"},
        # the package's headline frame: 1080p into the 512^3 caves
        {"name": "frame_1080p", "kind": "frame", "scene": "caves", "size": 512, "dim": 16,
         "width": 1920, "height": 1080, "fields": "view"},
        # a 4K frame of a large landscape
        {"name": "frame_4k", "kind": "frame", "scene": "heights", "size": 1024, "dim": 16,
         "width": 3840, "height": 2160, "fields": "view"},
        # a shaded preview in a window of odd size
        {"name": "shaded_window", "kind": "shaded", "scene": "caves", "size": 256, "dim": 8,
         "width": 1275, "height": 717, "convention": 0},
        # a frame at a level of detail
        {"name": "lod_1080p", "kind": "lod_frame", "scene": "caves", "size": 256, "dim": 16,
         "width": 1920, "height": 1080, "distance": 256.0, "fields": "view"},
        # secondary rays of one bounce of a small image
        {"name": "cast_300k", "kind": "cast", "scene": "caves", "size": 256, "dim": 8,
         "rays": 300007, "fields": "all"},
        # a large incoherent ray set (ambient occlusion, radiance probes)
        {"name": "cast_3m", "kind": "cast", "scene": "spheres", "size": 512, "dim": 32,
         "rays": 3000001, "fields": "view"},
        # level-of-detail queries of an incoherent set
        {"name": "lod_cast_500k", "kind": "lod_cast", "scene": "caves", "size": 128, "dim": 8,
         "rays": 500009, "distance": 128.0, "fields": "all"},
        # eight 1080p poses in one batched run: the package's headline step
        {"name": "batch_8x1080p", "kind": "batch", "scene": "caves", "size": 512, "dim": 16,
         "trees": 1, "views": 8, "width": 1920, "height": 1080},
        # many small trees with views of mixed sizes in one batched run
        {"name": "batch_mixed", "kind": "batch", "scene": "mixed", "size": 256, "dim": 0,
         "trees": 12, "views": 24, "width": 0, "height": 0},
        # an editor's step: change voxels, bring the device tree up to date,
        # look, take the change back, look again
        {"name": "edit_200", "kind": "edit", "scene": "caves", "size": 256, "dim": 8,
         "edits": 200, "width": 320, "height": 240},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "shaded", "lod_frame", "cast", "cast", "lod_cast",
                       "batch", "batch", "edit"])
    scene, size, dim = rng.choice([
        ("hills", 64, 4), ("hills", 128, 8), ("caves", 128, 8), ("caves", 256, 4),
        ("caves", 256, 16), ("caves", 512, 16), ("heights", 256, 4), ("heights", 512, 8),
        ("heights", 1024, 16), ("spheres", 512, 32)])
    if kind.startswith("lod"):
        scene, size, dim = rng.choice([("hills", 64, 4), ("hills", 128, 8), ("caves", 128, 8),
                                       ("caves", 128, 4), ("heights", 256, 8)])
    case = {"kind": kind, "scene": scene, "size": size, "dim": dim}
    if kind in ("frame", "shaded", "lod_frame", "edit"):
        pixels = _log_int(rng, 64 * 64, 3840 * 2160 if kind != "edit" else 640 * 480)
        aspect = rng.uniform(0.75, 2.4)
        case["width"] = max(8, int(math.sqrt(pixels * aspect)))
        case["height"] = max(8, int(math.sqrt(pixels / aspect)))
    if kind in ("cast", "lod_cast"):
        case["rays"] = _log_int(rng, 1, 3000000)
    if kind in ("frame", "lod_frame", "cast", "lod_cast"):
        case["fields"] = rng.choice(["all", "view"])
    if kind.startswith("lod"):
        case["distance"] = float(size) * rng.choice([0.25, 1.0, 4.0])
    if kind == "shaded":
        case["convention"] = rng.randrange(2)
    if kind == "edit":
        case["edits"] = _log_int(rng, 1, 200)
        if case["size"] > 256:
            case.update(scene="caves", size=256, dim=16)
    if kind == "batch":
        if rng.random() < 0.5:
            case.update(scene="mixed", size=rng.choice([128, 256, 512]), dim=0,
                        trees=rng.randint(2, 16), views=rng.randint(2, 32), width=0, height=0)
        else:
            case.update(trees=1, views=rng.randint(1, 8), width=rng.randint(64, 1920),
                        height=rng.randint(64, 1080))
    return case


# --- inputs ------------------------------------------------------------------


def _rng(seed):
    return np.random.default_rng(int(seed) % (1 << 31) + 17)


def _hills(size, seed):
    """A rolling landscape: voxel coordinates (n, 3) and packed colours."""
    rng = _rng(seed)
    ax = np.arange(size) / size
    h = np.zeros((size, size))
    for octave in range(1, 5):
        px, pz = rng.uniform(0, 2 * math.pi, 2)
        h += (np.sin(2 * math.pi * octave * ax + px)[:, None]
              + np.sin(2 * math.pi * octave * ax + pz)[None, :]) / octave
    h = ((h - h.min()) / (h.max() - h.min()) * 0.45 + 0.05) * size
    top = h.astype(np.int64)
    y = np.arange(size)[None, :, None]
    solid = (y < top[:, None, :]) & (y >= top[:, None, :] - 4)
    x, y, z = np.nonzero(solid)
    g = (y * 200 // size + 40).astype(np.uint32)
    colors = (np.uint32(60) << 24) | (g << np.uint32(16)) | (np.uint32(50) << 8) | np.uint32(255)
    return np.stack([x, y, z], 1).astype(np.uint32), colors, solid


def _octree(scene, size, dim, seed):
    if scene != "hills":
        return Octree.scene(SCENES[scene], size, dim, int(seed) % (1 << 31))
    tree = Octree(size, dim)
    xyz, colors, _ = _hills(size, seed)
    entries = np.zeros((len(xyz), 3), np.uint32)
    entries[:, 0] = 1
    entries[:, 1] = colors
    tree.insert_many(xyz, entries)
    return tree


def _view(size, width, height, rng):
    """(eye, direction, glass width, glass height), all f32 values: an eye on a
    circle around the tree, a little above it, a 60 degree lens."""
    f = np.float32
    c = size / 2.0
    a = rng.uniform(0, 2 * math.pi)
    eye = np.array([c + 1.2 * size * math.cos(a), 0.8 * size, c + 1.2 * size * math.sin(a)], f)
    d = np.array([c, 0.4 * size, c]) - eye
    d = (d / np.linalg.norm(d)).astype(f)
    gh = f(2 * math.tan(math.radians(30)))
    return eye, d, f(gh * f(width / height)), gh


def _viewport(view):
    eye, d, gw, gh = view
    return Viewport(tuple(float(v) for v in eye), tuple(float(v) for v in d),
                    (float(gw), float(gh), 1e9), 1.0)


def _rays(case, seed):
    """(n, 6) f32 origins and directions. Over hills: from the air towards the
    ground; elsewhere origins uniform in the tree, directions uniform."""
    n, size = case["rays"], case["size"]
    g = torch.Generator(device="cpu").manual_seed(int(seed) + 5)
    o = torch.rand((n, 3), generator=g, dtype=torch.float32) * size
    z = torch.rand((n,), generator=g, dtype=torch.float64) * 2 - 1
    phi = torch.rand((n,), generator=g, dtype=torch.float64) * (2 * math.pi)
    if case["scene"] == "hills":
        o[:, 1] = size * (0.55 + 0.4 * o[:, 1] / size)
        z = -z.abs()
    s = torch.sqrt(1 - z * z)
    d = torch.stack([s * torch.cos(phi), z, s * torch.sin(phi)], 1)
    d = (d / d.norm(dim=1, keepdim=True)).to(torch.float32)
    return torch.cat([o, d], 1)


def _views_of(case, rng):
    """[(tree, width, height)] of a batch."""
    if case["scene"] != "mixed":
        return [(0, case["width"], case["height"])] * case["views"]
    out = []
    for i in range(case["views"]):
        w, h = RESOLUTIONS[i % len(RESOLUTIONS)]
        out.append((i % case["trees"], w, h))
    return out


def _trees_of(case, seed):
    """[(scene, size, dim)] of a batch: sizes over 64 up to case["size"]."""
    if case["scene"] != "mixed":
        return [(case["scene"], case["size"], case["dim"])]
    steps = int(math.log2(case["size"])) - 5
    return [(("caves", "heights")[i % 2], 64 << (i % steps), (4, 8, 16)[i % 3])
            for i in range(case["trees"])]


def prepare(case, seed):
    kind, rng = case["kind"], _rng(seed)
    s = {"case": case}
    if kind == "batch":
        s["trees"] = [DeviceTree(_octree(sc, sz, dim, seed * 64 + i))
                      for i, (sc, sz, dim) in enumerate(_trees_of(case, seed))]
        sizes = [sz for _, sz, _ in _trees_of(case, seed)]
        views = _views_of(case, rng)
        # one array a field holds the images of all views, one after another
        s["image"] = alloc_hits(sum(w * h for _, w, h in views), "cuda", FIELDS["view"])
        s["jobs"], at = [], 0
        for t, w, h in views:
            bufs = {k: v[at:at + w * h] for k, v in s["image"].items()}
            at += w * h
            s["jobs"].append(Batch.render_job(s["trees"][t],
                                              _viewport(_view(sizes[t], w, h, rng)), w, h, bufs))
        s["batch"] = Batch(len(s["jobs"]))
        return s
    tree = _octree(case["scene"], case["size"], case["dim"], seed)
    if kind.startswith("lod"):
        tree.albedo_mip_map_resampling_strategy().switch_albedo_mip_maps(True).recalculate_mips()
    s["device"] = DeviceTree(tree)
    if "rays" in case:
        s["rays"] = _rays(case, seed).cuda()
    else:
        s["viewport"] = _viewport(_view(case["size"], case["width"], case["height"], rng))
    if kind == "frame" or kind == "edit":
        # a program that draws frame after frame keeps its image
        s["image"] = alloc_hits(case["width"] * case["height"], "cuda",
                                FIELDS[case.get("fields", "view")])
    if kind == "edit":
        s["tree"] = tree
        s["second"] = alloc_hits(case["width"] * case["height"], "cuda", FIELDS["view"])
        n = case["edits"]
        xyz = rng.integers(0, case["size"], (n, 3)).astype(np.uint32)
        entries = np.zeros((n, 3), np.uint32)
        entries[:, 0] = 1
        entries[:, 1] = rng.choice([0xC04020FF, 0x30A050FF, 0x5060F0FF, 0xE0E040FF], n)
        s["xyz"], s["entries"] = xyz, entries
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "cast":
        return s["device"].cast(s["rays"], FIELDS[case["fields"]])
    if kind == "lod_cast":
        return s["device"].cast_at_lod(s["rays"], case["distance"], FIELDS[case["fields"]])
    if kind == "batch":
        s["batch"].run(s["jobs"])
        return s["image"]
    w, h = case["width"], case["height"]
    if kind == "shaded":
        return s["device"].render_rgba8(s["viewport"], w, h, case["convention"])
    if kind == "lod_frame":
        return s["device"].render_at_lod(s["viewport"], w, h, case["distance"],
                                         FIELDS[case["fields"]])
    if kind == "edit":
        s["tree"].insert_many(s["xyz"], s["entries"])
        s["device"].update(s["tree"])
        s["device"].render_into(s["viewport"], w, h, s["image"])
        s["tree"].clear_many(s["xyz"])
        s["device"].update(s["tree"])
        s["device"].render_into(s["viewport"], w, h, s["second"])
        return {"after_insert": s["image"], "after_clear": s["second"]}
    s["device"].render_into(s["viewport"], w, h, s["image"])
    return s["image"]


def work(case):
    """Rays in, results out (which part of the tree a ray reads depends on the
    data: not counted), and the rays' own arithmetic."""
    kind = case["kind"]
    if kind == "batch":
        rays = sum(w * h for _, w, h in _views_of(case, None))
    else:
        rays = case["rays"] if "rays" in case else case["width"] * case["height"]
    per_ray = 4 if kind == "shaded" else sum(BYTES[k] for k in FIELDS[case.get("fields", "view")])
    if "rays" in case:
        per_ray += 24
    if kind == "edit":
        rays *= 2
    return {"bytes": float(rays * per_ray + 24 * 2 * case.get("edits", 0)),
            "flops": float(rays * FLOPS_PER_RAY)}


# --- 64-bit reference ----------------------------------------------------------


def _march(solid, o, d):
    """First solid voxel along each ray (f64): hit mask, distance, impact and
    the face normal, by voxel-to-voxel stepping through the dense grid."""
    size = solid.shape[0]
    n = len(o)
    with np.errstate(divide="ignore", invalid="ignore"):
        lo, hi = (0.0 - o) / d, (size - o) / d
    near, far = np.minimum(lo, hi).max(1), np.maximum(lo, hi).min(1)
    t = np.maximum(near, 0.0)
    live = (near <= far) & (far >= 0)
    axis = np.where(near > 0, np.minimum(lo, hi).argmax(1), -1)
    step = np.where(d < 0, -1, 1)
    p = o + d * t[:, None]
    cell = np.clip(np.floor(p).astype(np.int64), 0, size - 1)
    with np.errstate(divide="ignore", invalid="ignore"):
        tnext = (cell + (step > 0) - o) / d
        tdelta = np.abs(1.0 / d)
    hit = np.zeros(n, bool)
    while live.any():
        i = np.nonzero(live)[0]
        found = solid[cell[i, 0], cell[i, 1], cell[i, 2]]
        hit[i[found]] = True
        live[i[found]] = False
        i = i[~found]
        a = tnext[i].argmin(1)
        t[i] = tnext[i, a]
        axis[i] = a
        tnext[i, a] += tdelta[i, a]
        cell[i, a] += step[i, a]
        live[i[((cell[i] < 0) | (cell[i] >= size)).any(1)]] = False
    impact = np.where(hit[:, None], o + d * t[:, None], 0.0)
    normal = np.zeros((n, 3))
    faced = hit & (axis >= 0)
    normal[faced, axis[faced]] = -step[faced, axis[faced]]
    return hit, np.where(hit, t, np.inf), impact, normal


def exact(case, seed):
    """Distance, impact point and normal of frames and casts over the hills,
    whose voxels are known here. The package's scene generators, levels of
    detail and shading conventions are defined by their own f32 steps and have
    no other value; those cases return None."""
    if case["scene"] != "hills" or case["kind"] not in ("frame", "cast"):
        return None
    if case.get("rays", case.get("width", 1) * case.get("height", 1)) > 600000:
        return None
    size = case["size"]
    _, _, solid = _hills(size, seed)
    if case["kind"] == "cast":
        r = _rays(case, seed).numpy().astype(np.float64)
        o, d = r[:, :3], r[:, 3:]
    else:
        w, h = case["width"], case["height"]
        eye, look, gw, gh = (np.float64(v) for v in _view(size, w, h, _rng(seed)))
        up = np.array([0.0, 1.0, 0.0])
        right = np.cross(up, look)
        right /= np.linalg.norm(right)
        x = ((np.arange(w) + 0.5) / w - 0.5) * gw
        y = ((np.arange(h) + 0.5) / h - 0.5) * gh
        d = (look + x[None, :, None] * right + y[:, None, None] * up).reshape(-1, 3)
        d /= np.linalg.norm(d, axis=1, keepdims=True)
        o = np.broadcast_to(eye, d.shape)
    hit, t, impact, normal = _march(solid, o, d)
    values = {"distance": t, "impact": impact, "normal": normal}
    return {k: values.get(k) for k in FIELDS[case["fields"]]}
