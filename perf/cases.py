"""Performance cases: the calls a program makes through this package's entry points.

Meshes are perturbed spheres (icospheres and ragged latitude/longitude grids,
a few thousand to 1.3 million faces), seen from cameras around them, as in the
package's benchmark scenes. ``listed()`` names the cases, ``draw()`` gives more
of the same ranges, ``prepare()`` builds what a program holds before the call,
``run()`` is one call, ``exact()`` the call's float outputs in float64 from
plain torch.
"""
import functools
import math

import numpy as np
import torch

from ugu_amd import (ColorInterpolation, DiffuseColor, DiffuseShading, Rasterizer, Raytracer,
                     RendererCpuOption, ShadingNormal, _abi, scenes)
from ugu_amd.diff import DiffRenderer
from ugu_amd.texturing import texture_map_faces
from ugu_amd.types import Image1b, Image1f, Image1i, Image3b, Image3f, Mesh
from ugu_amd.visibility import Keyframe, VisibilityTester

PLANES = {"color": (3, torch.uint8), "depth": (0, torch.float32), "normal": (3, torch.float32),
          "mask": (0, torch.uint8), "face_id": (0, torch.int32)}


def listed():
    return [
        # a preview or thumbnail of a small mesh, vertex colours: launch latency
        dict(name="raster_small", kind="raster", stacks=128, slices=128, views=1, width=640,
             height=480, color="vertex", interp="bilinear", shading="none", normal="vertex",
             tex=0, tune=False),
        # the reference's own call: Render into host images, odd size, shaded texture
        dict(name="render_host", kind="render", stacks=205, slices=201, views=1, width=801,
             height=603, color="texture", interp="nn", shading="lambertian", normal="face",
             tex=512, tune=False),
        # one full-HD view of a scan-sized mesh with a texture
        dict(name="raster_1080p", kind="raster", level=8, views=1, width=1920, height=1080,
             color="texture", interp="bilinear", shading="none", normal="vertex", tex=2048,
             tune=True),
        # the headline workload: 64 views of mixed size in one call
        dict(name="raster_64_views", kind="raster", level=8, views=64, width=0, height=0,
             color="texture", interp="bilinear", shading="none", normal="vertex", tex=2048,
             tune=True),
        # the raytracer on the same full-HD view
        dict(name="raytrace_1080p", kind="raytrace", level=8, views=1, width=1920, height=1080,
             color="texture", interp="bilinear", shading="none", normal="vertex", tex=2048,
             tune=False),
        # the raytracer on many mixed views of a ragged mesh, shaded
        dict(name="raytrace_24_views", kind="raytrace", stacks=401, slices=613, views=24, width=0,
             height=0, color="vertex", interp="nn", shading="lambertian", normal="vertex", tex=0,
             tune=False),
        # face-wise visibility of a mesh in one keyframe (texturing a scan)
        dict(name="visibility_facewise", kind="visibility", level=7, width=1280,
             height=720),
        # writing a texture atlas from keyframes
        dict(name="texture_map", kind="texmap", level=6, views=8, width=640, height=480, tex=1024,
             padding=3),
        # one training view of a 100k-face mesh: colours, texture and positions
        dict(name="fit_one_view", kind="diff", stacks=225, slices=225, views=1, width=512,
             height=512, params="vertices+colors+texture", tex=1024),
        # a training step over 64 views: colours, texture and positions
        dict(name="fit_64_views", kind="diff", level=8, views=64, width=0, height=0,
             params="vertices+colors+texture", tex=2048),
        # inverse texturing: 32 views, the texture alone is learned
        dict(name="fit_texture_32_views", kind="diff", level=8, views=32, width=-1, height=-1,
             params="texture", tex=2048),
        # shape fitting without texture: positions and colours, odd view size
        dict(name="fit_shape_6_views", kind="diff", stacks=301, slices=407, views=6, width=799,
             height=601, params="vertices+colors", tex=0),
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    faces = log(2000, 1300000)
    ratio = rng.uniform(0.6, 1.6)
    stacks = max(8, int(math.sqrt(faces / 2 * ratio)))
    c = dict(stacks=stacks, slices=max(8, faces // (2 * stacks)))
    c["width"] = log(160, 1920)
    c["height"] = max(120, min(1080, int(c["width"] * rng.uniform(0.5, 0.9))))
    kind = rng.choice(["raster", "raster", "render", "raytrace", "raytrace", "visibility",
                       "texmap", "diff", "diff", "diff"])
    views = min(log(1, 64), 20_000_000 // (c["width"] * c["height"]))
    if kind == "visibility":
        c["stacks"], c["slices"] = min(c["stacks"], 401), min(c["slices"], 433)
        return dict(c, kind=kind)
    if kind == "texmap":
        c["stacks"], c["slices"] = min(c["stacks"], 301), min(c["slices"], 301)
        return dict(c, kind=kind, views=min(12, views), tex=log(200, 2048),
                    padding=rng.choice([1, 3, 5]))
    if kind == "diff":
        params = rng.choice(["vertices+colors+texture", "vertices+colors", "texture",
                             "colors+texture"])
        return dict(c, kind=kind, views=min(32, views), params=params,
                    tex=log(128, 2048) if "texture" in params else 0)
    if kind == "render":
        views = 1
    color = rng.choice(["texture", "texture", "vertex", "none"])
    return dict(c, kind=kind, views=views, color=color, interp=rng.choice(["nn", "bilinear"]),
                shading=rng.choice(["none", "lambertian", "oren-nayar"]),
                normal=rng.choice(["face", "vertex"]),
                tex=log(128, 2048) if color == "texture" else 0,
                tune=kind == "raster" and rng.random() < 0.5)


# --------------------------------------------------------------------------
# inputs


def _rng(seed, what):
    return np.random.default_rng([int(seed), what])


def _rand(shape, seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 64 + what)
    return torch.rand(shape, generator=g, device="cuda")


@functools.lru_cache(maxsize=4)
def _unit(level, stacks, slices):
    """Unit sphere: an icosphere, or a grid of stacks x slices quads with poles
    that are rings of their own (every row has slices + 1 vertices, u = 0..1)."""
    if level:
        v, f = scenes.icosphere_unit(level)
        phi = np.arctan2(v[:, 2], v[:, 0])
        uv = np.stack([phi / (2 * math.pi) + 0.5, 1 - np.arccos(np.clip(v[:, 1], -1, 1)) / math.pi],
                      1)
        return v, f.astype(np.int32), uv.astype(np.float32)
    i, j = np.meshgrid(np.arange(stacks + 1), np.arange(slices + 1), indexing="ij")
    theta = math.pi * (0.002 + 0.996 * i / stacks)
    phi = 2 * math.pi * j / slices
    v = np.stack([np.sin(theta) * np.cos(phi), np.cos(theta), np.sin(theta) * np.sin(phi)], -1)
    uv = np.stack([j / slices, 1 - i / stacks], -1)
    a = (np.arange(stacks)[:, None] * (slices + 1) + np.arange(slices)[None]).reshape(-1)
    b, c, d = a + 1, a + slices + 2, a + slices + 1
    f = np.stack([np.stack([a, b, c], 1), np.stack([a, c, d], 1)], 1).reshape(-1, 3)
    return v.reshape(-1, 3), f.astype(np.int32), uv.reshape(-1, 2).astype(np.float32)


def _mesh(case, seed):
    """Sphere of radius 1 + 0.05 sin(6 theta + a) cos(8 phi + b), a and b from the seed."""
    unit, faces, uv = _unit(case.get("level", 0), case.get("stacks", 0), case.get("slices", 0))
    a, b = _rng(seed, 0).uniform(0, 2 * math.pi, 2)
    theta = np.arccos(np.clip(unit[:, 1], -1, 1))
    phi = np.arctan2(unit[:, 2], unit[:, 0])
    r = 1 + 0.05 * np.sin(6 * theta + a) * np.cos(8 * phi + b)
    m = Mesh((unit * r[:, None]).astype(np.float32), faces)
    v = torch.from_numpy(m.vertices).cuda().double()[torch.from_numpy(faces).cuda().long()]
    n = torch.linalg.cross(v[:, 1] - v[:, 0], v[:, 2] - v[:, 0])
    # outward, whichever way the faces of the unit sphere wind
    if float((n * v.sum(1)).sum()) < 0:
        m.vertex_indices = np.ascontiguousarray(faces[:, [0, 2, 1]])
        n = -n
    n = n / n.norm(dim=1, keepdim=True).clamp_min(1e-30)
    m.set_face_normals(n.float().cpu().numpy())
    m.set_normals(unit.astype(np.float32))
    m.set_normal_indices(m.vertex_indices)
    m.set_uv(uv)
    m.set_uv_indices(m.vertex_indices)
    return m


def _sizes(case):
    n, w, h = case.get("views", 1), case["width"], case["height"]
    if w > 0:
        return [(w, h)] * n
    if w < 0:
        return [(512, 512)] * (n // 2) + [(1024, 768)] * (n - n // 2)
    pick = np.random.default_rng(2).integers(0, len(scenes.RES_CHOICES), n)
    return [scenes.RES_CHOICES[i] for i in pick]


def _cameras(case, seed):
    cams = []
    for k, size in enumerate(_sizes(case)):
        one = scenes.ring_cameras(max(2, case.get("views", 1)), 3.0, int(seed) + 1, 0, [size])
        cams.append(one[k])
    return cams


def _texture(case, seed):
    """Noise plus a 64-texel checker, float32 in [0, 1]."""
    s = case["tex"]
    k = torch.arange(s, device="cuda") // 64
    checker = ((k[:, None] + k[None]) % 2).float()[..., None]
    return 0.5 * _rand((s, s, 3), seed, 1) + 0.5 * checker


def _option(case):
    return RendererCpuOption(
        diffuse_color={"none": DiffuseColor.kNone, "texture": DiffuseColor.kTexture,
                       "vertex": DiffuseColor.kVertex}[case["color"]],
        interp={"nn": ColorInterpolation.kNn, "bilinear": ColorInterpolation.kBilinear}[
            case["interp"]],
        shading_normal={"face": ShadingNormal.kFace, "vertex": ShadingNormal.kVertex}[
            case["normal"]],
        diffuse_shading={"none": DiffuseShading.kNone, "lambertian": DiffuseShading.kLambertian,
                         "oren-nayar": DiffuseShading.kOrenNayar}[case["shading"]])


def _outputs(sizes):
    """One flat tensor per plane, and every view's part of it."""
    px = [w * h for w, h in sizes]
    flat = {k: torch.empty(sum(px) * max(1, c), dtype=t, device="cuda")
            for k, (c, t) in PLANES.items()}
    bufs, at = [], 0
    for (w, h), n in zip(sizes, px):
        bufs.append({k: flat[k][at * max(1, c):(at + n) * max(1, c)].view(
            (h, w, c) if c else (h, w)) for k, (c, _) in PLANES.items()})
        at += n
    return flat, bufs


def _keyframe(mesh, cam, seed):
    """Colour (smooth noise), depth and mask of the mesh in a view."""
    w, h = cam.width, cam.height
    low = _rand((1, 3, h // 16 + 2, w // 16 + 2), seed, 2)
    img = torch.nn.functional.interpolate(low, size=(h, w), mode="bilinear")[0].permute(1, 2, 0)
    view = _View(cam)
    fid, _ = view.visible(*_device(mesh))
    z = torch.zeros(h * w, device="cuda")
    on = (fid > 0).nonzero()[:, 0]
    z[on] = view.weights(_device(mesh)[0], _device(mesh)[1], fid[on], on)[1].float()
    return Keyframe(0, (img * 255).to(torch.uint8).cpu().numpy(), z.view(h, w).cpu().numpy(),
                    ((fid > 0).view(h, w) * 255).to(torch.uint8).cpu().numpy(), cam)


def _tex_faces(mesh, cams, tex):
    """Every face's record for the view that faces it most: its projected
    corners there and its uv triangle in texel coordinates."""
    p = mesh.vertices[mesh.vertex_indices]
    pos = np.stack([c.c2w[:3, 3] for c in cams])
    best = np.argmax(mesh.face_normals.astype(np.float64) @ pos.T, 1)
    src = np.zeros((len(p), 3, 2), np.float32)
    for k, c in enumerate(cams):
        on = best == k
        q = p[on].astype(np.float64) @ c.w2c[:3, :3].T + c.w2c[:3, 3]
        src[on] = q[..., :2] / q[..., 2:] * c.focal_length + c.principal_point
    uv = mesh.uv[mesh.uv_indices].astype(np.float64)
    wrap = uv[..., 0].max(1) - uv[..., 0].min(1) > 0.5
    uv[wrap, :, 0] += uv[wrap, :, 0] < 0.5
    rec = np.zeros(len(p), np.dtype([("keyframe", np.int32), ("src", np.float32, 6),
                                     ("dst", np.float32, 6)]))
    rec["keyframe"] = best
    rec["src"] = src.reshape(-1, 6)
    rec["dst"] = (np.stack([uv[..., 0], 1 - uv[..., 1]], -1) * tex - 0.5).reshape(-1, 6)
    return (_abi.UguTexFace * len(rec)).from_buffer(rec)


def prepare(case, seed):
    kind = case["kind"]
    mesh, cams = _mesh(case, seed), _cameras(case, seed)
    s = {"kind": kind, "cams": cams}
    if kind in ("raster", "render", "raytrace"):
        if case["color"] == "texture":
            mesh.set_single_material((_texture(case, seed) * 255).to(torch.uint8).cpu().numpy())
        if case["color"] == "vertex":
            mesh.set_vertex_colors(_rng(seed, 3).random((len(mesh.vertices), 3),
                                                        np.float32) * 255)
        r = s["renderer"] = (Raytracer if kind == "raytrace" else Rasterizer)(_option(case))
        r.set_mesh(mesh)
        assert r.PrepareMesh()
        if case["tune"]:
            r.autotune(cams, repeats=3)
        if kind == "render":
            r.set_camera(cams[0])
        else:
            s["flat"], bufs = _outputs(_sizes(case))
            s["binding"] = r.bind_device(cams, bufs)
    elif kind == "visibility":
        t = s["tester"] = VisibilityTester()
        t.set_data(mesh.vertices, mesh.normals, mesh.vertex_indices)
        assert t.PrepareData()
        t.set_keyframe(_keyframe(mesh, cams[0], seed))
        s["items"] = t.facewise_items()
    elif kind == "texmap":
        s["images"] = [(_rand((h, w, 3), seed, 8 + k) * 255).to(torch.uint8).cpu().numpy()
                       for k, (w, h) in enumerate(_sizes(case))]
        s["faces"] = _tex_faces(mesh, cams, case["tex"])
        s["tex"], s["padding"] = case["tex"], case["padding"]
    else:
        s["renderer"] = DiffRenderer(mesh)
        s["cams"] = [c.to_abi() for c in cams]
        s.update(_parameters(mesh, case, seed))
    return s


def _parameters(mesh, case, seed):
    p = {"vertices": torch.from_numpy(mesh.vertices).cuda(), "colors": None, "texture": None}
    if "colors" in case["params"]:
        p["colors"] = _rand((len(mesh.vertices), 3), seed, 4)
    if "texture" in case["params"]:
        p["texture"] = _texture(case, seed)
    learn = case["params"].split("+")
    for k in learn:
        p[k].requires_grad_(True)
    px = sum(w * h for w, h in _sizes(case))
    # dL/dimage of an image loss: signed, small
    return {"params": p, "learn": learn, "grad": (_rand(px * 3, seed, 5) - 0.5) * 0.1}


# --------------------------------------------------------------------------
# one pass


def run(s):
    kind = s["kind"]
    if kind in ("raster", "raytrace"):
        s["renderer"].render_bound(s["binding"])
        return dict(s["flat"])
    if kind == "render":
        img = [Image3b(), Image1f(), Image3f(), Image1b(), Image1i()]
        assert s["renderer"].Render(*img)
        return {k: i.data for k, i in zip(PLANES, img)}
    if kind == "visibility":
        rec, _ = s["tester"].test_items(*s["items"])
        return {k: rec[k] for k in rec.dtype.names}
    if kind == "texmap":
        tex, mask = texture_map_faces(s["images"], s["faces"], len(s["faces"]), s["tex"],
                                      s["tex"], s["padding"])
        return {"texture": tex, "mask": mask}
    p = s["params"]
    image, fid = s["renderer"].render_flat(s["cams"], p["vertices"], p["colors"], p["texture"])
    grads = torch.autograd.grad(image, [p[k] for k in s["learn"]], s["grad"])
    return {"image": image, "face_id": fid, **{"grad_" + k: g for k, g in zip(s["learn"], grads)}}


def work(case):
    """Inputs once and outputs once; operations: about 60 per (face, view), 40 per
    pixel, for gradients 500 float64 per pixel."""
    if case.get("level"):
        F = 20 * 4 ** case["level"]
        V = F // 2 + 2
    else:
        F = 2 * case["stacks"] * case["slices"]
        V = (case["stacks"] + 1) * (case["slices"] + 1)
    px = sum(w * h for w, h in _sizes(case))
    n, kind = case.get("views", 1), case["kind"]
    mesh = 12 * V + 12 * F
    tex = case.get("tex", 0) ** 2
    if kind == "visibility":
        return {"bytes": mesh + 3 * F * 36 + 3 * F * 36 + 8 * px, "flops": 3 * F * 400}
    if kind == "texmap":
        return {"bytes": 52 * F + 3 * px + 4 * tex, "flops": 60 * F + 40 * tex}
    if kind == "diff":
        b = mesh + (8 * V + 12 * F + 12 * tex if tex else 0)
        for k, size in (("vertices", 12 * V), ("colors", 24 * V), ("texture", 12 * tex)):
            b += size if k in case["params"] else 0
        return {"bytes": 2 * mesh + b + 32 * px, "flops": 60 * F * n + 540 * px}
    b = mesh + 12 * F
    b += 12 * V + 12 * F if case["normal"] == "vertex" else 0
    b += {"none": 0, "vertex": 12 * V, "texture": 8 * V + 16 * F + 3 * tex}[case["color"]]
    return {"bytes": b + 24 * px, "flops": 60 * F * n + 40 * px}


# --------------------------------------------------------------------------
# float64 results


def _device(mesh):
    return (torch.from_numpy(mesh.vertices).cuda(),
            torch.from_numpy(mesh.vertex_indices).cuda().long(),
            torch.from_numpy(mesh.face_normals).cuda())


def _spread(counts):
    """For counts n_i: i repeated n_i times, and 0..n_i - 1 within each."""
    i = torch.repeat_interleave(torch.arange(len(counts), device=counts.device), counts)
    return i, torch.arange(len(i), device=counts.device) - (counts.cumsum(0) - counts)[i]


def _sum3(a):
    return a[..., 0] + (a[..., 1] + a[..., 2])


def _edge(a, b, c):
    return (c[0] - a[0]) * (b[1] - a[1]) - (c[1] - a[1]) * (b[0] - a[0])


def _unit_rows(v):
    n = _sum3(v * v)
    return torch.where(n[..., None] > 0, v / n.sqrt()[..., None], v)


class _View:
    """A camera's float32 numbers and what is computed with them: which face a
    pixel shows (float32, the renderer's comparisons) and its weights (float64)."""

    def __init__(self, cam):
        abi = cam.to_abi()
        t = lambda x, *s: torch.tensor(list(x), dtype=torch.float32, device="cuda").view(*s)  # noqa: E731
        self.w, self.h = abi.width, abi.height
        self.f = t([abi.fx, abi.fy], 2)
        self.c = t([abi.cx, abi.cy], 2)
        self.R, self.t = t(abi.w2c_R, 3, 3), t(abi.w2c_t, 3)
        self.Rc, self.o = t(abi.c2w_R, 3, 3), t(abi.c2w_t, 3)

    def project(self, v):
        q = _sum3(self.R.to(v) * v[..., None, :]) + self.t.to(v)
        xy = self.f.to(v) / q[..., 2:] * q[..., :2] + self.c.to(v)
        return torch.cat([xy, q[..., 2:]], -1)

    def rays(self, xy):
        d = (xy - self.c.to(xy)) / self.f.to(xy)
        d = _unit_rows(torch.cat([d, torch.ones_like(d[:, :1])], 1))
        return _sum3(self.Rc.to(xy) * d[:, None, :])

    def pixel(self, pix, dtype):
        return torch.stack([pix % self.w, pix // self.w], 1).to(dtype)

    def candidates(self, p, margin=0.0):
        """(face, pixel) pairs of the faces' pixel boxes; p: F x 3 x 3 projected."""
        lo = torch.ceil(p[..., :2].amin(1) - margin).clamp(min=0)
        hi = torch.floor(p[..., :2].amax(1) + margin)
        hi = torch.minimum(hi, torch.tensor([self.w - 1, self.h - 1], device="cuda").to(hi))
        n = (hi - lo + 1).clamp(min=0).long()
        face, k = _spread(n[:, 0] * n[:, 1])
        x = lo[face, 0].long() + k % n[face, 0]
        y = lo[face, 1].long() + k // n[face, 0]
        return face, y * self.w + x

    def nearest(self, face, pix, depth):
        """Per pixel the face of the smallest float32 depth, the lowest face on ties."""
        key = (depth.float().view(torch.int32).long() << 32) | face
        none = 2 ** 63 - 1
        best = torch.full((self.w * self.h,), none, dtype=torch.long, device="cuda")
        best.scatter_reduce_(0, pix, key, "amin")
        return torch.where(best < none, best & 0xffffffff, torch.full_like(best, -1))

    def visible(self, verts, faces, fn):
        """Face id per pixel (-1: none or culled), and whether the winner faces away."""
        p = self.project(verts)[faces]
        face, pix = self.candidates(p)
        q = p[face]
        a, b, c = ((q[:, k, 0], q[:, k, 1]) for k in range(3))
        xy = self.pixel(pix, torch.float32)
        x = (xy[:, 0], xy[:, 1])
        every = self.rays(self.pixel(torch.arange(self.w * self.h, device="cuda"), torch.float32))
        away = _sum3(fn[face] * every[pix]) > 0
        e = torch.stack([_edge(b, c, x), _edge(c, a, x), _edge(a, b, x)], 1)
        area = _edge(a, b, c)
        on = torch.where(away, (e <= 0).all(1), (e >= 0).all(1)) & (q[..., 2] >= 0).all(1)
        on &= area.abs() >= torch.finfo(torch.float32).tiny
        e = e / area[:, None] / q[..., 2]
        z = 1 / ((e[:, 0] + e[:, 1]) + e[:, 2])
        fid = self.nearest(face[on], pix[on], z[on])
        back = (fid >= 0) & (_sum3(fn[fid.clamp(min=0)] * every) > 0)
        return torch.where(back, torch.full_like(fid, -1), fid), back

    def weights(self, verts, faces, fid, pix):
        """Perspective-correct weights and depth in float64 of pixels `pix` showing `fid`."""
        q = self.project(verts.double()[faces[fid]])
        a, b, c = ((q[:, k, 0], q[:, k, 1]) for k in range(3))
        xy = self.pixel(pix, torch.float64)
        x = (xy[:, 0], xy[:, 1])
        e = torch.stack([_edge(b, c, x), _edge(c, a, x), _edge(a, b, x)], 1)
        e = e / _edge(a, b, c)[:, None] / q[..., 2]
        z = 1 / e.sum(1)
        return e * z[:, None], z

    def traced(self, verts, faces, fn):
        """Face id, weights and distance per pixel of the nearest ray-triangle hit."""
        p = self.project(verts.double())[faces]
        face, pix = self.candidates(p, 0.01)
        ray = self.rays(self.pixel(pix, torch.float32)).double()
        hit, t, w = _intersect(verts.double()[faces[face]], self.o.double(), ray)
        fid = self.nearest(face[hit], pix[hit], t[hit])
        on = (fid >= 0).nonzero()[:, 0]
        ray = self.rays(self.pixel(on, torch.float32))
        on = on[_sum3(fn[fid[on]] * ray) <= 0]
        ray = self.rays(self.pixel(on, torch.float32)).double()
        _, t, w = _intersect(verts.double()[faces[fid[on]]], self.o.double(), ray)
        return on, fid[on], w, (self.o.double() + ray * t[:, None])


def _intersect(v, o, d):
    """Ray-triangle test: hit, distance and the corners' weights."""
    e1, e2, r = v[:, 1] - v[:, 0], v[:, 2] - v[:, 0], o - v[:, 0]
    al, be = torch.linalg.cross(d, e2), torch.linalg.cross(r, e1)
    det = (e1 * al).sum(1)
    u, w, t = (al * r).sum(1) / det, (be * d).sum(1) / det, (be * e2).sum(1) / det
    hit = (det.abs() >= 1e-8) & (u >= 0) & (w >= 0) & (u + w <= 1) & (t >= 0)
    return hit, t, torch.stack([1 - u - w, u, w], 1)


def _exact_render(case, seed):
    mesh = _mesh(case, seed)
    verts, faces, fn = _device(mesh)
    depth, normal = [], []
    for cam in _cameras(case, seed):
        v = _View(cam)
        z = torch.zeros(v.w * v.h, dtype=torch.float64, device="cuda")
        n = torch.zeros(v.w * v.h, 3, dtype=torch.float64, device="cuda")
        if case["kind"] == "raytrace":
            on, fid, w, hit = v.traced(verts, faces, fn)
            z[on] = hit @ v.R[2].double() + v.t[2].double()
            # the raytracer's first two weights are those of corners 1 and 2 shifted by one:
            # (1 - u - v, u, v) multiply corners (0, 1, 2) with u, v the weights of 0 and 1
            w = torch.stack([w[:, 2], w[:, 0], w[:, 1]], 1)
        else:
            fid, _ = v.visible(verts, faces, fn)
            keep = (fid >= 0).nonzero()[:, 0]
            z[keep] = v.weights(verts, faces, fid[keep], keep)[1]
            on = (fid > 0).nonzero()[:, 0]
            fid = fid[on]
            w, _ = v.weights(verts, faces, fid, on)
        if case["normal"] == "face":
            m = fn[fid].double()
        else:
            m = (w[..., None] * torch.from_numpy(mesh.normals).cuda().double()[faces[fid]]).sum(1)
        n[on] = m @ v.R.double().T
        depth.append(z)
        normal.append(n.view(-1))
    out = {"color": None, "depth": torch.cat(depth), "normal": torch.cat(normal), "mask": None,
           "face_id": None}
    if case["kind"] == "render":
        w, h = _sizes(case)[0]
        out["depth"], out["normal"] = out["depth"].view(h, w), out["normal"].view(h, w, 3)
    return out


def _bilinear(tex, uv):
    h, w = tex.shape[:2]
    x, y = uv[:, 0] * (w - 1), (1 - uv[:, 1]) * (h - 1)
    fx, fy = x.detach().floor(), y.detach().floor()
    x0, y0 = fx.long(), fy.long()
    lu, lv = (x - fx)[:, None], (y - fy)[:, None]
    at = lambda i, j: tex[i.clamp(0, h - 1), j.clamp(0, w - 1)]  # noqa: E731
    return ((1 - lu) * (1 - lv) * at(y0, x0) + lu * (1 - lv) * at(y0, x0 + 1)
            + (1 - lu) * lv * at(y0 + 1, x0) + lu * lv * at(y0 + 1, x0 + 1))


def _exact_diff(case, seed):
    mesh = _mesh(case, seed)
    s = _parameters(mesh, case, seed)
    faces = torch.from_numpy(mesh.vertex_indices).cuda().long()
    uv = torch.from_numpy(mesh.uv).cuda().double()
    p = {k: None if v is None else v.detach().double() for k, v in s["params"].items()}
    leaves = [p[k].requires_grad_(True) for k in s["learn"]]
    v32 = s["params"]["vertices"].detach()
    t = v32[faces]
    e1, e2 = _unit_rows(t[:, 1] - t[:, 0]), _unit_rows(t[:, 2] - t[:, 0])
    fn = torch.stack([e1[:, 1] * e2[:, 2] - e1[:, 2] * e2[:, 1],
                      e1[:, 2] * e2[:, 0] - e1[:, 0] * e2[:, 2],
                      e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0]], 1)
    fn = _unit_rows(fn)
    total = [torch.zeros_like(x) for x in leaves]
    images, at = [], 0
    for cam in _cameras(case, seed):
        v = _View(cam)
        n = v.w * v.h
        with torch.no_grad():
            fid, _ = v.visible(v32, faces, fn)
            on = (fid > 0).nonzero()[:, 0]
        w, _ = v.weights(p["vertices"], faces, fid[on], on)
        c = torch.ones(len(on), 3, dtype=torch.float64, device="cuda")
        if p["colors"] is not None:
            c = c * (w[..., None] * p["colors"][faces[fid[on]]]).sum(1)
        if p["texture"] is not None:
            c = c * _bilinear(p["texture"], (w[..., None] * uv[faces[fid[on]]]).sum(1))
        g = s["grad"][at * 3:(at + n) * 3].view(-1, 3)[on].double()
        for acc, got in zip(total, torch.autograd.grad(c, leaves, g)):
            acc += got
        img = torch.zeros(n, 3, dtype=torch.float64, device="cuda")
        img[on] = c.detach()
        images.append(img.view(-1))
        at += n
    return {"image": torch.cat(images), "face_id": None,
            **{"grad_" + k: g for k, g in zip(s["learn"], total)}}


def _exact_visibility(case, seed):
    """Projection and angle of the items a keyframe sees. Every item is a ray of
    its own: the faces it can meet are those over the item's pixel cell."""
    mesh = _mesh(case, seed)
    verts, faces, _ = _device(mesh)
    cam = _cameras(case, seed)[0]
    kf = _keyframe(mesh, cam, seed)
    v = _View(cam)
    v.R = torch.from_numpy(cam.w2c[:3, :3].astype(np.float32)).cuda()
    c = ((verts[faces][:, 0] + verts[faces][:, 1]) + verts[faces][:, 2]) / 3
    tri = verts[faces]
    pos = (tri + (c[:, None] - tri) * 1e-3).reshape(-1, 3)
    nrm = torch.from_numpy(mesh.normals).cuda()[faces].reshape(-1, 3)
    p = v.project(pos.double())
    xy = p[:, :2]
    ok = (p[:, 2] >= 0) & (xy >= 0).all(1) & (xy[:, 0] <= v.w - 1) & (xy[:, 1] <= v.h - 1)
    near = xy.round().clamp(min=0).long()
    pix = (near[:, 1].clamp(max=v.h - 1) * v.w + near[:, 0].clamp(max=v.w - 1))
    ok &= torch.from_numpy(kf.mask).cuda().view(-1)[pix] == 255
    ok &= torch.from_numpy(kf.depth).cuda().view(-1)[pix] >= 1.2e-7
    ray = v.rays(xy)
    angle = torch.acos(-(nrm.double() * ray).sum(1))
    ok &= angle <= math.pi / 2
    item = ok.nonzero()[:, 0]
    cell = xy[item, 1].floor().long() * v.w + xy[item, 0].floor().long()
    order = cell.argsort()
    item, cell = item[order], cell[order]
    first = torch.searchsorted(cell, torch.arange(v.w * v.h + 1, device="cuda"))
    q = v.project(verts.double())[faces]
    q[..., :2] = torch.stack([q[..., :2].amin(1).floor(), q[..., :2].amax(1).floor(),
                              q[..., :2].amax(1).floor()], 1)
    face, at = v.candidates(q)
    k, j = _spread(first[at + 1] - first[at])
    face, who = face[k], item[first[at[k]] + j]
    dist = torch.full((len(pos),), math.inf, dtype=torch.float64, device="cuda")
    hit, t, _ = _intersect(verts.double()[faces[face]], v.o.double(), ray[who])
    dist.scatter_reduce_(0, who[hit], t[hit], "amin")
    gap = (v.o.double() + ray * dist[:, None] - tri.reshape(-1, 3).double()).norm(dim=1)
    # a ray that slips past every face occludes nothing (and has the largest float as distance)
    ok &= torch.isinf(dist) | (gap <= 0.1)
    pick = lambda x, off: torch.where(ok, x, torch.full_like(x, off))  # noqa: E731
    return {"visible": None, "px": pick(xy[:, 0], 0.0), "py": pick(xy[:, 1], 0.0),
            "angle": pick(angle, float(np.float32(999.9))), "dist": None, "c0": None, "c1": None,
            "c2": None, "intensity": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "texmap":
        return None  # bytes
    if kind == "visibility":
        return _exact_visibility(case, seed)
    return _exact_diff(case, seed) if kind == "diff" else _exact_render(case, seed)
