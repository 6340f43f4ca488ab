"""The work that programs have this render core do, as cases to be timed and compared.

listed() names the cases, draw(rng) gives more of the same ranges, prepare(case,
seed) makes what a program holds before the call (a context with its scene built,
device buffers, options), run(state) is one pass through aurora_amd's public entry
points and returns its outputs, work(case) is what a pass cannot do without and
exact(case, seed) the outputs' values in 64 bits where they can be had.

Kinds of case:
  closest, any  standalone traversal of device ray buffers;
  rebuild       the tree build of uploaded geometry, and its permutation (which
                maps hit ids back to the caller's triangles);
  pbr, compat   a whole frame, copied out to the caller's device buffer;
  diff          one differentiable-rendering step: forward image, backward to the
                albedos and radiances;
  batch         many preview jobs of different scenes in one call.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from aurora_amd import diff, native, scenes

DEV = "cuda"
SPHERE_TRIS = 20  # an icosphere has 20 * 4^subdivisions triangles


def listed() -> list[dict]:
    return [
        # a probe query: a few rays into a small scene (picking, light probes)
        {"name": "closest-probe", "kind": "closest", "scene": "cornell", "size": 2, "rays": "incoherent", "n": 1000},
        # the headline workload: incoherent rays into 1,024,002 triangles
        {"name": "closest-incoherent-1M", "kind": "closest", "scene": "spheres", "size": 200, "rays": "incoherent",
         "n": 1 << 24},
        # camera rays of a full-HD frame, the first query of any ray caster
        {"name": "closest-camera-1M", "kind": "closest", "scene": "spheres", "size": 200, "rays": "camera",
         "n": 1920 * 1080},
        # visibility segments between points of the scene (shadows, occlusion)
        {"name": "any-segments-1M", "kind": "any", "scene": "spheres", "size": 200, "rays": "segments",
         "n": 1_000_003},
        # a scene far larger than the caches
        {"name": "closest-soup-10M", "kind": "closest", "scene": "soup", "size": 10_000_000, "rays": "incoherent",
         "n": 1 << 21},
        # an edit of a small scene: rebuild before the next frame
        {"name": "rebuild-cornell", "kind": "rebuild", "scene": "cornell", "size": 2},
        # a scene load, or a deforming mesh's rebuild per frame
        {"name": "rebuild-1M", "kind": "rebuild", "scene": "spheres", "size": 200},
        # an interactive preview of a small scene
        {"name": "pbr-cornell", "kind": "pbr", "scene": "cornell", "size": 2, "width": 256, "height": 256,
         "spp": 16, "depth": 4},
        # a step of a full-HD progressive render of a large scene
        {"name": "pbr-1M-1080p", "kind": "pbr", "scene": "spheres", "size": 200, "width": 1920, "height": 1080,
         "spp": 8, "depth": 8},
        # the reference's own estimator (drop-in mode), an odd frame size
        {"name": "compat-1M", "kind": "compat", "scene": "spheres", "size": 200, "width": 1279, "height": 719,
         "spp": 4, "depth": 8},
        # an optimisation step of the differentiable renderer
        {"name": "diff-cornell", "kind": "diff", "scene": "c5", "size": 20, "width": 512, "height": 512, "spp": 4,
         "depth": 6},
        # a farm of preview renders
        {"name": "batch-16", "kind": "batch", "scene": "c4", "size": 16, "width": 256, "spp": 16, "depth": 6},
    ]


def _log(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["closest", "closest", "any", "rebuild", "pbr", "compat", "diff", "batch"])
    scene = rng.choice(["cornell", "spheres", "soup"])
    size = {"cornell": _log(rng, 1, 40), "spheres": _log(rng, 1, 200), "soup": 2 * _log(rng, 1, 1_000_000)}[scene]
    if kind in ("closest", "any"):
        rays = "segments" if kind == "any" else rng.choice(["incoherent", "incoherent", "camera"])
        return {"kind": kind, "scene": scene, "size": size, "rays": rays, "n": _log(rng, 1, 1 << 22)}
    if kind == "rebuild":
        return {"kind": kind, "scene": scene, "size": size}
    if kind == "batch":
        return {"kind": kind, "scene": "c4", "size": rng.randint(1, 16), "width": rng.choice([64, 128, 256]),
                "spp": rng.choice([1, 4, 16]), "depth": rng.randint(1, 8)}
    w, h = _log(rng, 16, 1920), _log(rng, 16, 1080)
    if kind == "diff":
        w, h = min(w, 640), min(h, 640)
        return {"kind": kind, "scene": "c5", "size": rng.randint(2, 20), "width": w, "height": h,
                "spp": rng.choice([1, 2, 4]), "depth": rng.randint(1, 8)}
    scene = rng.choice(["cornell", "spheres"])
    return {"kind": kind, "scene": scene, "size": _log(rng, 1, 40 if scene == "cornell" else 200), "width": w,
            "height": h, "spp": rng.randint(1, 8), "depth": rng.randint(1, 8)}


# ---- scenes and rays, from the seed alone


def _soup(n: int, seed: int) -> scenes.Scene:
    """scenes.soup's distribution (equilateral triangles, edge ~ LogNormal(0, 1),
    random orientation, uniform centroids), made on the GPU: 10M triangles take
    seconds on the host.  The box keeps scenes.soup's density (10M in 1000^3)."""
    g = torch.Generator(DEV).manual_seed(seed)
    box = 1000.0 * (n / 10_000_000) ** (1.0 / 3.0)
    c = torch.rand((n, 1, 3), generator=g, device=DEV) * box
    edge = torch.exp(torch.randn((n, 1, 1), generator=g, device=DEV))
    a = torch.nn.functional.normalize(torch.randn((n, 3), generator=g, device=DEV), dim=1)
    b = torch.nn.functional.normalize(torch.cross(a, torch.randn((n, 3), generator=g, device=DEV), dim=1), dim=1)
    corner = torch.tensor([[1.0, 0.0], [-0.5, math.sqrt(3) / 2], [-0.5, -math.sqrt(3) / 2]], device=DEV) / math.sqrt(3)
    P = c + edge * (corner[None, :, :1] * a[:, None] + corner[None, :, 1:] * b[:, None])  # (n, 3 corners, 3)
    v = P.transpose(1, 2).reshape(n, 9)
    nrm = torch.cross(a, b, dim=1).repeat(1, 3)
    base = scenes.random_soup(1, 2)
    cam = scenes.make_camera((0.5 * box, 0.5 * box, -0.6 * box), (0.0, 0.0, 1.0), (1.0, 1.0))
    return scenes.Scene(vertices=scenes.canonical(v.cpu().numpy()), normals=scenes.canonical(nrm.cpu().numpy()),
                        texcoords=np.zeros((n, 6), np.float32), shader_ids=np.ones(n, np.uint16),
                        shaders=base.shaders, lights=base.lights, camera=cam, name=f"soup-{n}")


def _scene(case: dict, seed: int) -> scenes.Scene:
    w, h = case.get("width", 1920), case.get("height", 1080)
    if case["scene"] == "cornell":
        return scenes.cornell(seed=seed, n_spheres=case["size"], subdivisions=3, width=w, height=h)
    if case["scene"] == "spheres":
        return scenes.spheres(seed=seed, n_spheres=case["size"], width=w, height=h)
    if case["scene"] == "c5":
        return scenes.cornell(seed=seed, n_spheres=case["size"], subdivisions=4, width=w, height=h, n_lights=4,
                              split_materials=True)
    return _soup(case["size"], seed)


def _box(case: dict) -> float:
    if case["scene"] == "cornell":
        return 5.0
    return 100.0 if case["scene"] == "spheres" else 1000.0 * (case["size"] / 10_000_000) ** (1.0 / 3.0)


def _rays(case: dict, scene: scenes.Scene, seed: int) -> torch.Tensor:
    """(n, 8) float32 ray records: origin, tmax, direction, 0."""
    n, box = case["n"], _box(case)
    g = torch.Generator(DEV).manual_seed(seed + 1)
    rays = torch.zeros((n, 8), device=DEV)
    rays[:, 3] = 1_000_000.0
    if case["rays"] == "camera":  # pixel-ordered pinhole rays of a 16:9 frame, the last row cut
        w = max(1, int(math.sqrt(n * 16 / 9)))
        h = (n + w - 1) // w
        i = torch.arange(n, device=DEV)
        cam = {k: torch.tensor(np.array(scene.camera[k]), device=DEV) for k in ("position", "right", "up", "forward")}
        t = [float(x) for x in scene.camera["tanfov"]]
        off = torch.rand(2, generator=g, device=DEV)
        px, py = ((i % w) + off[0]) / w - 0.5, ((i // w) + off[1]) / h - 0.5
        d = px[:, None] * cam["right"] * t[0] + py[:, None] * cam["up"] * t[1] + cam["forward"]
        rays[:, 0:3] = cam["position"]
        rays[:, 4:7] = torch.nn.functional.normalize(d, dim=1)
        return rays
    rays[:, 0:3] = torch.rand((n, 3), generator=g, device=DEV) * box
    if case["rays"] == "segments":
        d = torch.rand((n, 3), generator=g, device=DEV) * box - rays[:, 0:3]
        length = d.norm(dim=1)
        rays[:, 3] = length
        rays[:, 4:7] = d / length[:, None]
        return rays
    u = torch.rand((n, 2), generator=g, device=DEV)
    z = 1.0 - 2.0 * u[:, 0]
    r = torch.sqrt(torch.clamp(1.0 - z * z, min=0.0))
    rays[:, 4], rays[:, 5], rays[:, 6] = r * torch.cos(2 * math.pi * u[:, 1]), r * torch.sin(2 * math.pi * u[:, 1]), z
    return rays


# ---- the state a program holds, and one pass


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "diff":
        scene = _scene(case, seed)
        g = torch.Generator(DEV).manual_seed(seed)
        s["renderer"] = diff.DiffRenderer(scene, case["spp"], case["depth"], seed=seed & 0x7FFFFFFF)
        s["albedo"] = torch.tensor(scene.shaders["diffuse_color"] * scene.shaders["diffuse"][:, None], device=DEV,
                                   requires_grad=True)
        s["radiance"] = torch.tensor(scene.lights["color"] * scene.lights["intensity"][:, None], device=DEV,
                                     requires_grad=True)
        s["target"] = torch.rand((scene.width * scene.height, 3), generator=g, device=DEV)
        torch.cuda.synchronize()
        return s
    ctx = s["ctx"] = native.Context(0)
    if kind == "batch":
        # Cornell scenes with 2..40 spheres as scenes.c4_jobs makes them, two sizes and sample counts
        jobs = [scenes.cornell(seed=(seed + k) & 0x7FFFFFFF, n_spheres=2 + (13 * k) % 39, subdivisions=4,
                               width=case["width"] >> (k % 2), height=case["width"] >> (k % 2),
                               spp=case["spp"] if k % 3 else max(1, case["spp"] // 4)) for k in range(case["size"])]
        specs = [{"scene": ctx.scene_add(j), "width": j.width, "height": j.height, "spp": j.spp,
                  "max_depth": case["depth"], "rr_start": 3, "seed": (seed + k) & 0x7FFFFFFF, "camera": j.camera}
                 for k, j in enumerate(jobs)]
        s["jobs"] = native.Context.make_jobs(specs)
        s["out"] = torch.zeros((sum(j.width * j.height for j in jobs), 4), device=DEV)
        torch.cuda.synchronize()
        return s
    scene = _scene(case, seed)
    ctx.upload_scene(scene)
    if kind == "rebuild":
        return s
    ctx.rebuild_nmh()
    if kind in ("closest", "any"):
        s["rays"] = _rays(case, scene, seed)
        s["out"] = (torch.zeros((case["n"], 4), device=DEV) if kind == "closest"
                    else torch.zeros(case["n"], dtype=torch.int32, device=DEV))
    else:
        ctx.frame_create(case["width"], case["height"], case["spp"])
        s["camera"] = scene.camera
        s["opts"] = native.Context.opts(native.MODE_PBR if kind == "pbr" else native.MODE_COMPAT, case["spp"],
                                        case["depth"], 3, seed & 0x7FFFFFFF)
        s["out"] = torch.zeros((case["width"] * case["height"], 4), device=DEV)
    torch.cuda.synchronize()
    return s


def run(s: dict):
    kind = s["kind"]
    if kind == "diff":
        image = diff.render(s["renderer"], s["albedo"], s["radiance"])
        loss = torch.mean((image - s["target"]) ** 2)
        grads = torch.autograd.grad(loss, [s["albedo"], s["radiance"]])
        return {"image": image.detach(), "albedo": grads[0], "radiance": grads[1]}
    ctx = s["ctx"]
    if kind == "closest":
        ctx.trace_closest_ptr(s["rays"].shape[0], s["rays"].data_ptr(), s["out"].data_ptr())
        return {"id": s["out"].view(torch.int32)[:, 0], "tuv": s["out"][:, 1:]}
    if kind == "any":
        ctx.trace_any_ptr(s["rays"].shape[0], s["rays"].data_ptr(), s["out"].data_ptr())
        return {"id": s["out"]}
    if kind == "rebuild":
        ctx.rebuild_nmh()
        return {"permutation": ctx.read_permutation().view(np.int32)}
    if kind == "batch":
        ctx.batch_render_ptr(s["jobs"], s["out"].data_ptr())
        return {"images": s["out"]}
    ctx.frame_render(s["camera"], s["opts"])
    ctx.frame_copy_ptr(s["out"].data_ptr())
    return {"image": s["out"]}


# ---- what a pass cannot do without


def _triangles(case: dict) -> int:
    k = case["size"]
    return {"cornell": 24 + k * SPHERE_TRIS * 64, "spheres": 2 + k * SPHERE_TRIS * 256,
            "c5": 24 + k * SPHERE_TRIS * 256, "soup": k, "c4": 24 + 21 * SPHERE_TRIS * 256}[case["scene"]]


def work(case: dict) -> dict:
    """bytes: inputs once, outputs once.  flops: a ray's node visits, about 2.2
    per tree level (44.8 at 19 levels, measured), at 2 triangle tests (54 each)
    and two slab tests; a path's rays: one extension and its next-event rays per
    bounce, a third of the bounces survive a hit."""
    tris, kind = _triangles(case), case["kind"]
    levels = max(1, math.ceil(math.log2(max(2, tris / 2))))
    visit = 2 * 54 + 16
    if kind in ("closest", "any"):
        n = case["n"]
        touched = min(48 * tris, 48 * 2.2 * levels * n)
        return {"bytes": n * (48 if kind == "closest" else 36) + touched, "flops": n * 2.2 * levels * visit}
    if kind == "rebuild":
        # vertices, normals, uvs and ids read and written, the records and the permutation written
        return {"bytes": tris * (2 * 98 + 48 + 4), "flops": tris * levels * 4}
    pixels = case["width"] * (case["width"] if kind == "batch" else case["height"])
    jobs = case["size"] if kind == "batch" else 1
    lights = {"spheres": 4, "c5": 4}.get(case["scene"], 1)
    paths = pixels * jobs * case["spp"] * (0.47 if kind == "batch" else 1.0)
    bounces = 2.0 if kind == "compat" else 1 + 0.35 * (case["depth"] - 1)
    rays = paths * bounces * (1 + lights) * (2 if kind == "diff" else 1)
    return {"bytes": 48 * tris * jobs + 16 * pixels * jobs, "flops": rays * 2.2 * levels * visit}


def exact(case: dict, seed: int):
    """Closest hits by testing every triangle (one-sided Moller-Trumbore) in
    64 bits; ids follow the tree's order, so they have no value of their own.
    Images and gradients are estimates of integrals that plain code cannot
    repeat draw by draw."""
    if case["kind"] != "closest" or case["n"] * _triangles(case) > 4_000_000_000:
        return None
    scene = _scene(case, seed)
    rays = _rays(case, scene, seed).double()
    v = torch.from_numpy(scene.vertices).to(DEV).double().reshape(-1, 3, 3).transpose(1, 2)  # (m, corner, xyz)
    v1, e1, e2 = v[:, 0], v[:, 1] - v[:, 0], v[:, 2] - v[:, 0]
    normal, area = torch.cross(e1, e2, dim=1), 1e-7
    out = torch.zeros((case["n"], 3), dtype=torch.float64, device=DEV)
    step = max(1, 16_000_000 // v.shape[0])
    for s in range(0, case["n"], step):
        o, tmax, d = rays[s : s + step, 0:3], rays[s : s + step, 3], rays[s : s + step, 4:7]
        det = -(d @ normal.T)
        T = o[:, None, :] - v1[None]
        C = torch.cross(T, d[:, None, :].expand_as(T), dim=2)  # T x d
        u = (C * e2[None]).sum(2) / det
        w = (C * e1[None]).sum(2) / -det
        t = (T * normal[None]).sum(2) / det
        u, w, t = (torch.where(det < area, torch.full_like(t, float("inf")), x) for x in (u, w, t))
        ok = (u >= 0) & (w >= 0) & (u + w <= 1) & (t > 1e-7) & (t < tmax[:, None])
        best = torch.where(ok, t, torch.full_like(t, float("inf")))
        t_min, k = best.min(dim=1)
        hit = torch.isfinite(t_min)
        pick = torch.arange(o.shape[0], device=DEV)
        out[s : s + step, 0] = torch.where(hit, t_min, tmax)
        out[s : s + step, 1] = torch.where(hit, u[pick, k], torch.zeros_like(t_min))
        out[s : s + step, 2] = torch.where(hit, w[pick, k], torch.zeros_like(t_min))
    return {"id": None, "tuv": out}
