"""What a user of the renderer has it do, as cases that can be timed and compared.

A case is a scene family, an entry point and its sizes:

* ``cube``        a null-BSDF cube holding a heterogeneous fBm medium, a quad light and an
                  emissive enclosing sphere: the benchmark's scene;
* ``dielectric``  a displaced rough-dielectric sphere of 25K to 100K faces inside a
                  heterogeneous medium, two lights, one tangent lane per deformation;
* ``surface``     a diffuse icosphere over a ground quad, no media;
* ``glass``       a rough-dielectric ball over a ground quad, no media, translation lanes
                  and one roughness lane: the shape of the glass_1 example.

Entry points (``path``): ``ad`` VolPathTracerAD, ``path_ad`` PathTracerAD, ``direct_ad``
DirectAD, ``primal`` VolPathTracer, ``simple`` VolPathTracerSimple, ``path`` PathTracer,
``particles`` ParticleTracer, ``density`` the differentiable density render (forward image
and the gradient of every grid node), ``views`` several uneven views in one call and
``step`` one inverse-rendering step over several views. All are Monte Carlo estimates
over the renderer's own counter-based streams, so no value of theirs can be had without
restating the whole estimator: ``exact`` gives none.
"""
import functools
import math

import numpy as np
import torch
import torch.nn.functional as F

import dtrt_amd.dtrt as dtrt
from dtrt_amd import adjoint, scenes
from dtrt_amd.scenes import MediumDesc, SceneDesc, ShapeDesc

KIND = {"ad": 0, "primal": 1, "simple": 2, "path": 3, "particles": 5, "path_ad": 6, "direct_ad": 7}
INTERIOR = 1 | 2 | 8   # EMode bits of the terms the density adjoint differentiates


def _case(scene, path, **kw):
    c = dict(scene=scene, path=path, nder=3, width=64, height=64, spp=16, depth=10, sppe=4096, sppse=10, grid=64,
             faces=0, views=1, bits=64)
    c.update(kw)
    return c


def listed():
    def named(name, *a, **kw):
        return dict(_case(*a, **kw), name=name)
    return [
        # a preview of a few samples: launches, host round trips and the longest path
        named("cube_preview", "cube", "ad", width=32, height=32, spp=4),
        # one small view of an optimisation that renders many
        named("cube_view", "cube", "ad", width=128, height=128, spp=16),
        # the benchmark render, at its full size
        named("cube_full", "cube", "ad", width=512, height=512, spp=128),
        # the same scene with the single-precision kernel set, odd width, spp not a multiple of a wave
        named("cube_float", "cube", "ad", width=333, height=250, spp=48, bits=32),
        # many tangent lanes on a large mesh in a medium: the refilling kernels, deep paths
        named("dielectric_lanes8", "dielectric", "ad", nder=8, width=192, height=192, spp=16, depth=12, grid=128,
              faces=100000),
        # surfaces only, one lane: interface edges and primary edges
        named("surface_lane1", "surface", "ad", nder=1, width=256, height=256, spp=64, depth=5, grid=0),
        # the optimisation example's shape: rough dielectric, four lanes, many primary-edge samples
        named("glass_lanes4", "glass", "ad", nder=4, width=256, height=256, spp=128, depth=4, sppe=4096, grid=0),
        # a density optimisation step: image forward, gradient of 128^3 nodes backward
        named("density_grad", "cube", "density", nder=1, width=512, height=512, spp=32, sppe=0, sppse=0, grid=128),
        # a target image
        named("cube_primal", "cube", "primal", width=512, height=512, spp=64),
        # light tracing of the same scene
        named("cube_particles", "cube", "particles", width=256, height=256, spp=32),
        # eight uneven views in one call
        named("cube_views8", "cube", "views", width=96, height=80, spp=16, views=8),
        # one inverse-rendering step: views, loss, lane gradients and the density adjoint
        named("dielectric_step", "dielectric", "step", nder=8, width=96, height=96, spp=8, depth=12, grid=128, faces=25000,
              views=3),
    ]


def draw(rng):
    """One more case of the same ranges; sizes over their logarithm."""
    def between(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def image(most, spp_lo, spp_hi):   # about `most` samples
        spp = between(spp_lo, min(spp_hi, most // 256))
        w = max(16, min(512, int(math.sqrt(most / spp) * rng.uniform(0.7, 1.4))))
        return dict(width=w, height=max(16, min(512, most // (spp * w))), spp=spp)
    kind = rng.choice(["cube", "cube", "cube", "dielectric", "surface", "glass", "density", "primal", "views", "step"])
    if kind == "cube":
        bits = rng.choice([64, 64, 32])
        return _case("cube", "ad", nder=rng.choice([1, 2, 3, 3, 4]), bits=bits, depth=rng.choice([4, 8, 10]),
                     sppse=rng.choice([4, 10]), grid=between(24, 128), **image(between(4096, 1 << 24), 4, 128))
    if kind == "dielectric":
        return _case("dielectric", "ad", nder=rng.choice([3, 4, 8, 8]), depth=rng.choice([6, 12]), grid=between(32, 128),
                     faces=between(5000, 100000), **image(between(4096, 1 << 19), 4, 64))
    if kind == "surface":
        return _case("surface", rng.choice(["ad", "path_ad", "direct_ad"]), nder=rng.choice([1, 3]), depth=5, grid=0,
                     **image(between(4096, 1 << 22), 4, 128))
    if kind == "glass":
        return _case("glass", "ad", nder=4, depth=4, sppe=between(1024, 4096), grid=0, **image(between(4096, 1 << 22), 8, 128))
    if kind == "density":
        return _case("cube", "density", nder=1, sppe=0, sppse=0, grid=between(32, 128), depth=rng.choice([5, 10]),
                     **image(between(16384, 1 << 22), 8, 64))
    if kind == "primal":
        scene, path = rng.choice([("cube", "primal"), ("cube", "simple"), ("dielectric", "primal"), ("surface", "path")])
        faces = 50000 if scene == "dielectric" else 0
        return _case(scene, path, depth=rng.choice([5, 10]), grid=0 if scene == "surface" else between(32, 128), faces=faces,
                     **image(between(16384, 1 << (20 if faces else 23)), 8, 128))
    if kind == "views":
        return _case("cube", "views", views=rng.randint(2, 8), **image(between(4096, 1 << 16), 4, 32))
    return _case("dielectric", "step", nder=8, depth=12, grid=between(32, 128), faces=between(5000, 25000),
                 views=rng.randint(1, 3), **image(between(2048, 1 << 16), 4, 16))


# ------------------------------------------------------------------------ scenes
def _fbm(res, seed):
    """Value-noise fBm on res^3 nodes, rescaled to [0, 2]."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = torch.zeros((1, 1, res, res, res), device="cuda")
    for octave in range(4):
        n = (4 << octave) + 1
        lattice = torch.rand((1, 1, n, n, n), generator=g, device="cuda")
        out += 0.5 ** octave * F.interpolate(lattice, size=(res, res, res), mode="trilinear", align_corners=True)
    lo, hi = out.min(), out.max()
    return (2.0 * (out - lo) / (hi - lo))[0, 0].cpu().numpy()


@functools.lru_cache(maxsize=None)
def _icosphere(subdiv, radius, center, inward=False):
    return scenes.icosphere(subdiv, radius, center, inward=inward)


def _sphere(faces):
    """Welded latitude-longitude sphere of about `faces` triangles, outward winding."""
    rows = max(4, int(round(math.sqrt(faces / 4.0))))
    cols = 2 * rows
    th = np.pi * np.arange(1, rows)[:, None] / rows
    ph = 2 * np.pi * np.arange(cols)[None, :] / cols
    ring = np.stack([np.sin(th) * np.cos(ph), np.cos(th) + 0 * ph, -np.sin(th) * np.sin(ph)], -1).reshape(-1, 3)
    v = np.concatenate([[[0.0, 1.0, 0.0]], ring, [[0.0, -1.0, 0.0]]])
    j = np.arange(cols)
    k = (j + 1) % cols
    top = np.stack([0 * j, 1 + j, 1 + k], -1)
    i = (1 + cols * np.arange(rows - 2))[:, None]
    a, b, c, d = i + j, i + k, i + cols + j, i + cols + k
    mid = np.concatenate([np.stack([a, c, d], -1).reshape(-1, 3), np.stack([a, d, b], -1).reshape(-1, 3)])
    last = 1 + cols * (rows - 2)
    bottom = np.stack([last + j, 0 * j + len(v) - 1, last + k], -1)
    return v, np.concatenate([top, mid, bottom]).astype(np.int32)


def _field(dirs, rng, terms=6):
    """A smooth scalar field on the unit sphere, in [-1, 1]."""
    out = np.zeros(len(dirs))
    for _ in range(terms):
        a = rng.normal(size=3)
        a /= np.linalg.norm(a)
        out += np.cos((1.0 + 3.0 * rng.random()) * np.pi * (dirs @ a) + 2 * np.pi * rng.random())
    return out / terms


def _cube(case, seed):
    n, moving = case["nder"], case["path"] != "density"
    c_v, c_f = scenes.cube()
    l_v, l_f = scenes.quad((0, 1.5, 0), 1.0, 1, -1)
    e_v, e_f = _icosphere(2, 20.0, (0, 0, 0), inward=True)
    vel, tvel = np.zeros((n, len(c_v), 3), np.float32), np.zeros((n, 3), np.float32)
    for k in range(min(n, 3)):
        vel[k, :, k] = tvel[k, k] = 1.0 if moving else 0.0
    med = MediumDesc("heterogeneous", density=_fbm(case["grid"], seed), trans_vel=tvel, rot_vel=np.zeros((n, 3), np.float32))
    return dict(shapes=[ShapeDesc(c_v, c_f, bsdf_id=0, med_int=0, velocities=vel), ShapeDesc(l_v, l_f, bsdf_id=1, light_id=0),
                        ShapeDesc(e_v, e_f, bsdf_id=1, light_id=1)],
                bsdfs=[("null",), ("diffuse", (0.0, 0.0, 0.0))],
                lights=[("area", 1, (20.0, 20.0, 20.0), False), ("area", 2, (0.5, 0.5, 0.5), True)],
                phases=[("hg", 0.3)], media=[med], edge_weights=np.array([1.0, 1.0, 0.0], np.float32)), (0, 0, 3)


def _dielectric(case, seed):
    n, rng = case["nder"], np.random.default_rng(seed)
    dirs, f = _sphere(case["faces"])
    v = (dirs * (0.5 + 0.03 * _field(dirs, rng)[:, None])).astype(np.float32)
    nrm = scenes.vertex_normals(v, f)
    vel = np.stack([(nrm * _field(dirs, rng)[:, None]).astype(np.float32) for _ in range(n)])
    c_v, c_f = scenes.cube(-1.0, 1.0)
    a_v, a_f = scenes.quad((0, 2.0, 0), 1.0, 1, -1)
    b_v, b_f = scenes.quad((2.0, 0.5, 0), 1.0, 0, -1)
    med = MediumDesc("heterogeneous", density=_fbm(case["grid"], seed), bmin=(-1, -1, -1), bmax=(1, 1, 1))
    return dict(shapes=[ShapeDesc(v, f, bsdf_id=2, med_ext=0, normals=nrm, velocities=vel),
                        ShapeDesc(c_v, c_f, bsdf_id=0, med_int=0), ShapeDesc(a_v, a_f, bsdf_id=1, light_id=0),
                        ShapeDesc(b_v, b_f, bsdf_id=1, light_id=1)],
                bsdfs=[("null",), ("diffuse", (0.0, 0.0, 0.0)), ("roughdielectric", 0.01, 1.5, 1.0)],
                lights=[("area", 2, (15.0, 15.0, 15.0), False), ("area", 3, (8.0, 8.0, 8.0), False)],
                phases=[("hg", 0.3)], media=[med]), (0, 0.3, 3.2)


def _surface(case, seed):
    n, rng = case["nder"], np.random.default_rng(seed)
    g_v, g_f = scenes.quad((0, 0, 0), 4.0, 1, +1)
    s_v, s_f = _icosphere(3, 0.5, (0, 0.5, 0))
    s_v = (s_v + rng.uniform(-0.2, 0.2, 3) * (1, 0, 1)).astype(np.float32)
    l_v, l_f = scenes.quad((0, 2.5, 0), 1.0, 1, -1)
    vel = np.zeros((n, len(s_v), 3), np.float32)
    for k in range(min(n, 3)):
        vel[k, :, k] = 1.0
    return dict(shapes=[ShapeDesc(g_v, g_f, bsdf_id=0), ShapeDesc(s_v, s_f, bsdf_id=1, velocities=vel),
                        ShapeDesc(l_v, l_f, bsdf_id=2, light_id=0)],
                bsdfs=[("diffuse", (0.5, 0.5, 0.5)), ("diffuse", (0.8, 0.8, 0.8)), ("diffuse", (0.0, 0.0, 0.0))],
                lights=[("area", 2, (10.0, 10.0, 10.0), False)]), (0, 1.5, 3.5)


def _glass(case, seed):
    n, rng = case["nder"], np.random.default_rng(seed)
    g_v, g_f = scenes.quad((0, 0, 0), 6.0, 1, +1)
    s_v, s_f = _icosphere(3, 0.6, (0, 0.8, 0))
    s_v = (s_v + rng.uniform(-0.2, 0.2, 3)).astype(np.float32)
    l_v, l_f = scenes.quad((0, 4.0, 0), 2.0, 1, -1)
    vel = np.zeros((n, len(s_v), 3), np.float32)
    for k in range(min(n, 3)):
        vel[k, :, k] = 1.0
    d_alpha = np.zeros(n, np.float32)
    d_alpha[-1] = 0.1
    return dict(shapes=[ShapeDesc(g_v, g_f, bsdf_id=0), ShapeDesc(s_v, s_f, bsdf_id=1, velocities=vel),
                        ShapeDesc(l_v, l_f, bsdf_id=2, light_id=0)],
                bsdfs=[("diffuse", (0.6, 0.5, 0.4)), ("roughdielectric", 0.2, 1.5, 1.0, d_alpha),
                       ("diffuse", (0.0, 0.0, 0.0))],
                lights=[("area", 2, (12.0, 12.0, 12.0), False)]), (0, 2.0, 5.0)


def _view_sizes(case):
    """Uneven sizes around the case's own, one per view."""
    return [(case["width"] * (4 + 5 * v % 8) // 6 + v, case["height"] * (4 + 3 * v % 8) // 6, case["spp"])
            for v in range(case["views"])]


def prepare(case, seed):
    parts, eye = {"cube": _cube, "dielectric": _dielectric, "surface": _surface, "glass": _glass}[case["scene"]](case, seed)
    ndc = scenes.cam_to_ndc(40.0)
    at = (0, 0, 0) if case["scene"] in ("cube", "dielectric") else (0, 0.5, 0)
    desc = SceneDesc(nder=case["nder"], width=case["width"], height=case["height"], cam_to_world=scenes.look_at(eye, at, (0, 1, 0)),
                     cam_to_ndc=ndc, spp=case["spp"], max_bounces=case["depth"], sppe=case["sppe"], sppse=case["sppse"], **parts)
    before = dtrt.precision()
    dtrt.set_precision(case["bits"])
    try:
        scene = scenes.instantiate(dtrt, desc)
    finally:
        dtrt.set_precision(before)
    path, forward = case["path"], case["path"] in ("ad", "path_ad", "direct_ad")
    mode = INTERIOR if path == "density" else -1
    s = dict(case=case, scene=scene, path=path,
             options=dtrt.RenderOptions(seed, case["spp"], case["depth"], case["sppe"], case["sppse"], True, mode, 0.0),
             shape=((case["nder"] + 1,) if forward else ()) + (case["height"], case["width"], 3))
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    if path == "density":
        s["density"] = torch.tensor(parts["media"][0].density, device="cuda", requires_grad=True)
        s["target"] = torch.rand(s["shape"], generator=g, device="cuda")
    if path in ("views", "step"):
        s["cameras"], s["view_options"], s["adjoint_options"], s["targets"] = [], [], [], []
        r = math.hypot(*eye)
        for v, (w, h, spp) in enumerate(_view_sizes(case)):
            phi, elev = 2 * math.pi * v / case["views"] + 0.1, 0.3 * math.sin(1.0 + v)
            pos = (r * math.cos(elev) * math.sin(phi), r * math.sin(elev), r * math.cos(elev) * math.cos(phi))
            s["cameras"].append(dtrt.Camera(w, h, scenes.look_at(pos, at, (0, 1, 0)), ndc, 1e-2, -1, None))
            s["view_options"].append(dtrt.RenderOptions(seed + v, spp, case["depth"], case["sppe"], case["sppse"], True, -1, 0.0))
            s["adjoint_options"].append(dtrt.RenderOptions(seed + 100 + v, spp, case["depth"], 0, 0, True, INTERIOR, 0.0))
            s["targets"].append(0.2 * torch.rand((h, w, 3), generator=g, device="cuda"))
        s["view_shapes"] = [(case["nder"] + 1, h, w, 3) for w, h, _ in _view_sizes(case)]
        s["grid_shape"] = (case["grid"],) * 3
    return s


def run(s):
    path = s["path"]
    if path in KIND:
        image = torch.zeros(s["shape"], device="cuda")
        dtrt.render_device(KIND[path], s["scene"], s["options"], image.data_ptr())
        return image
    if path == "density":
        s["density"].grad = None
        image = adjoint.render_density(s["density"], s["scene"], s["options"], (s["case"]["nder"] + 1,) + s["shape"])
        (image - s["target"]).pow(2).mean().backward()
        return {"image": image.detach(), "grad": s["density"].grad}
    images = [torch.zeros(sh, device="cuda") for sh in s["view_shapes"]]
    if path == "views":
        dtrt.render_views(s["scene"], s["cameras"], s["view_options"], images)
        return images
    grad = torch.zeros(s["grid_shape"], device="cuda")
    lanes = torch.zeros(s["case"]["nder"], dtype=torch.float64, device="cuda")
    loss = torch.zeros(1, dtype=torch.float64, device="cuda")
    dtrt.step(s["scene"], s["cameras"], s["view_options"], images, s["targets"], 0, s["adjoint_options"], grad, lanes, loss)
    return {"images": images, "density": grad, "lanes": lanes, "loss": loss}


def exact(case, seed):
    return None


# Operations of one sample: per scene those without tangents and those of one lane, from
# the renderer's own counts of the box tests (at 24 operations), triangle tests (45),
# density lookups (60) and hit records the estimator asks for on these scenes, sub-paths
# included; a primal sample needs a fraction of the first, having no sub-paths.
FLOPS = {"cube": (23000, 900), "dielectric": (75000, 5000), "surface": (56000, 500), "glass": (90000, 700)}
PRIMAL = {"cube": 0.15, "dielectric": 0.1, "surface": 0.1, "glass": 0.1}


def work(case):
    sizes = _view_sizes(case) if case["path"] in ("views", "step") else [(case["width"], case["height"], case["spp"])]
    pixels, samples = sum(w * h for w, h, _ in sizes), sum(w * h * n for w, h, n in sizes)
    per, lane = FLOPS[case["scene"]]
    n = case["nder"]
    tangents = n if case["path"] in ("ad", "path_ad", "direct_ad", "views", "step") else 0
    if case["path"] == "particles":
        samples = 100000 * case["spp"]
    if case["path"] in ("primal", "simple", "path", "particles", "density"):   # no sub-paths
        per *= PRIMAL[case["scene"]]
        lane *= 0.5
        tangents = 3 * n if case["path"] == "density" else 0   # forward, then both passes of the replay
    flops = samples * (per + lane * tangents)
    faces = {"cube": 334, "dielectric": case["faces"], "surface": 1284, "glass": 1284}[case["scene"]]
    lanes = n if case["path"] in ("ad", "path_ad", "direct_ad", "views", "step") else 0
    size = 4 * case["grid"] ** 3 + faces * (60 + 18 * n) + 12 * pixels * (1 + lanes)
    if case["path"] in ("density", "step"):
        size += 4 * case["grid"] ** 3 + 24 * pixels
    return {"bytes": float(size), "flops": float(flops)}
