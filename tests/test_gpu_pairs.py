"""Expansion of a tile's faces to (face, pixel) pairs, against the oracle at the
sizes where it can go wrong: faces of one pixel up to the whole tile, numbers of
faces and of pairs around a wavefront's 64 and a chunk's face slots, slivers whose
box holds many pixels they miss, and mixes of all of these in one tile. Face id,
mask and colour are exact, depth within 1e-5 (as in the parity tests)."""
import numpy as np
import pytest

import oracle as O
from ugu_amd import (DiffuseColor, Mesh, PinholeCamera, Rasterizer, Raytracer, RendererCpuOption,
                     ShadingNormal)

pytestmark = pytest.mark.gpu

W, H, F = 70, 45, 64.0  # ragged tiles in both directions


def _camera():
    return PinholeCamera(W, H, np.eye(4), (W * 0.5 - 0.5, H * 0.5 - 0.5), (F, F))


def _box(x, y, w, h, rng):
    """A triangle whose pixel box is about (x .. x + w - 1, y .. y + h - 1)."""
    p = np.array([[0, 0], [w, 0], [0, h]], float) - 0.5 + rng.uniform(0.01, 0.4, (3, 2))
    if rng.random() < 0.5:
        p = p[::-1] * [1, -1] + [0, h - 1]
    return p + [x, y]


def _sliver(x, y, n, rng):
    p = np.array([[0, 0], [n, n - 1], [n - 0.3, n - 1]], float) + rng.uniform(0, 0.2, (3, 2))
    return p * [1, rng.choice([-1, 1])] + [x, y]


def _scene(kind, rng):
    if kind == "one":
        return [_box(-300, -300, 900, 900, rng)]
    if kind.startswith("full"):  # every face over the first tile and beyond it
        return [_box(-40, -40, 200, 200, rng) for _ in range(int(kind[4:]))]
    if kind.startswith("px"):    # faces of a pixel or two, all in one tile
        return [_box(rng.integers(0, 7), rng.integers(0, 7), rng.integers(1, 3),
                     rng.integers(1, 3), rng) for _ in range(int(kind[2:]))]
    if kind == "slivers":
        return [_sliver(rng.uniform(-2, W), rng.uniform(0, H), rng.integers(3, 40), rng)
                for _ in range(200)]
    tris = []
    for _ in range(330):
        k = rng.integers(0, 5)
        x, y = rng.uniform(-3, W), rng.uniform(-3, H)
        if k == 0:
            tris.append(_sliver(x, y, rng.integers(3, 30), rng))
        else:
            n = [0, 1, 3, 9, 40][k]
            tris.append(_box(x, y, rng.integers(1, n + 1), rng.integers(1, n + 1), rng))
    return tris


KINDS = ["one", "full1", "full64", "full65", "full257", "px1", "px63", "px64", "px65", "px256",
         "px257", "px700", "slivers", "mix"]


def _mesh(kind):
    rng = np.random.default_rng(KINDS.index(kind))
    tris = np.stack(_scene(kind, rng))
    n = len(tris)
    z = (2.0 + rng.permutation(n) * 1e-3)[:, None] + rng.uniform(0, 0.2, (n, 3)) * (rng.random((n, 1)) < 0.5)
    cx, cy = W * 0.5 - 0.5, H * 0.5 - 0.5
    p = np.stack([(tris[..., 0] - cx) / F * z, (tris[..., 1] - cy) / F * z, z], -1)
    m = Mesh(p.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.int32))
    m.CalcFaceNormal()
    m.set_normals(np.repeat(m.face_normals, 3, axis=0))
    m.set_normal_indices(m.vertex_indices)
    m.set_vertex_colors(rng.random((3 * n, 3), np.float32) * 255)
    return m


def _option(culling):
    return RendererCpuOption(diffuse_color=DiffuseColor.kVertex, shading_normal=ShadingNormal.kFace,
                             backface_culling=culling)


def _equal(out, ref, label):
    for k in ("face_id", "mask", "color"):
        bad = np.argwhere(out[k] != ref[k])
        assert len(bad) == 0, (label, k, bad[:5])
    np.testing.assert_allclose(out["depth"], ref["depth"], rtol=1e-5, atol=0)


@pytest.mark.parametrize("kind", KINDS)
def test_rasterizer(gpu_available, kind):
    mesh, cam = _mesh(kind), _camera()
    for culling in (False, True):
        opt = _option(culling)
        rc, ref, _ = O.render(mesh, O.camera_from_abi(cam.to_abi()), opt, c2w_t=cam.c2w[:3, 3])
        assert rc == 0
        r = Rasterizer(opt)
        r.set_mesh(mesh)
        assert r.PrepareMesh()
        for tile in ((8, 8), (16, 16), (32, 8)):
            for persistent in (False, True):
                r.set_tiling(*tile, bin_capacity=64, persistent=persistent)
                views = [cam] * (1 if kind == "px1" else 2)
                for out in r.render_batch(views):
                    _equal(out, ref, (kind, tile, persistent, culling))


@pytest.mark.parametrize("kind", KINDS)
def test_raytracer(gpu_available, kind):
    mesh, cam, opt = _mesh(kind), _camera(), _option(False)
    rc, ref, _ = O.raytrace(mesh, O.camera_from_abi(cam.to_abi()), opt, c2w_t=cam.c2w[:3, 3])
    assert rc == 0
    r = Raytracer(opt)
    r.set_mesh(mesh)
    assert r.PrepareMesh()
    _equal(r.render_batch([cam])[0], ref, kind)
