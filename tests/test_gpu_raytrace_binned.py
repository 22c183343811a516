"""The raytracer's binned path and its hand-over to the hierarchy, against
oracle_raytrace (every face for every pixel, float64): poses whose linear part
is not a rotation, faces across the camera's plane, coordinates of any scale,
sub-pixel faces, and tiles whose bins grow or overflow. Every output but the
colour-independent floats is compared exactly; depth and normal within 1e-5
relative, the bound the raytracer's other parity tests use."""
import numpy as np
import pytest

import oracle as O
from ugu_amd import DiffuseColor, Mesh, PinholeCamera, Raytracer, RendererCpuOption, scenes

pytestmark = pytest.mark.gpu


def _soup(n, size, spread, seed, offset=(0.0, 0.0, 0.0)):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-spread, spread, (n, 1, 3)) + np.asarray(offset)
    v = (c + rng.uniform(-size, size, (n, 3, 3))).reshape(-1, 3)
    return _finish(Mesh(v.astype(np.float32), np.arange(3 * n, dtype=np.int32)), seed)


def _finish(m, seed):
    m.CalcFaceNormal()
    m.set_normals(np.repeat(m.face_normals, 3, axis=0)[:len(m.vertices)])
    m.set_normal_indices(m.vertex_indices)
    m.set_vertex_colors(np.random.default_rng(seed).random((len(m.vertices), 3), np.float32) * 255)
    return m


def _sphere(level):
    v, f = scenes.icosphere_unit(level)
    m = scenes.perturbed_sphere(v, f)
    m.set_vertex_colors(np.random.default_rng(1).random((len(m.vertices), 3), np.float32) * 255)
    return m


def _camera(w, h, linear=None, pos=(0.0, 0.0, -3.0), f=None):
    c2w = np.eye(4)
    if linear is not None:
        c2w[:3, :3] = linear
    c2w[:3, 3] = pos
    f = f or (0.9 * h, 0.9 * h)
    return PinholeCamera(w, h, c2w, (w * 0.5 - 0.5, h * 0.5 - 0.5), f)


def _layers(n, w):
    """n triangles over pixels around (8, 8) of a w x w view, a pixel or so each,
    and one far away (which keeps the mesh's mean number of layers low)."""
    rng = np.random.default_rng(n)
    z = rng.permutation(n)[:, None] * 1e-3 + 2.0
    uv = rng.uniform(-0.02, 0.02, (n, 1, 2)) + rng.uniform(-0.04, 0.04, (n, 3, 2))
    uv += (8 - (w * 0.5 - 0.5)) / (0.9 * w)
    p = np.concatenate([uv * z[..., None], np.repeat(z[..., None], 3, 1)], -1)
    p[..., 2] -= 3.0
    p[-1] += 60.0
    return _finish(Mesh(p.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.int32)), n)


def _forms():
    rot = np.linalg.qr(np.random.default_rng(4).normal(size=(3, 3)))[0]
    yield "rotation", _sphere(4), _camera(77, 45, rot, tuple(-3.0 * rot[:, 2]))
    yield "scaled", _sphere(3), _camera(64, 49, 1.7 * np.eye(3))
    yield "sheared", _sphere(3), _camera(50, 64, np.eye(3) + np.triu(np.full((3, 3), 0.2), 1))
    yield "ill_conditioned", _sphere(3), _camera(40, 40, np.diag([1.0, 1.0, 12.0]))
    yield "inside", _sphere(3), _camera(61, 47, pos=(0.1, 0.2, 0.0), f=(15.0, 19.0))
    yield "across_the_camera", _soup(150, 1.0, 1.5, 5), _camera(37, 53, pos=(0, 0, 0))
    yield "millimetres", _soup(200, 300.0, 900.0, 6, (0, 0, 1500.0)), _camera(48, 48)
    yield "far_away", _soup(200, 1e-3, 4e-3, 7, (50, -20, 900.0)), \
        _camera(64, 40, pos=(50, -20, 899.98))
    yield "negative_focal", _sphere(3), _camera(33, 31, f=(-30.0, 41.0))
    yield "sub_pixel", _sphere(5), _camera(17, 15)
    yield "one_pixel", _sphere(2), _camera(1, 1, f=(5.0, 5.0))
    yield "bins_grow", _layers(2500, 24), _camera(24, 24)
    yield "bins_overflow", _layers(6000, 24), _camera(24, 24)


@pytest.mark.parametrize("form", [f[0] for f in _forms()])
@pytest.mark.parametrize("culling", [False, True])
def test_binned_raytrace_matches_oracle(gpu_available, form, culling):
    _, mesh, cam = next(f for f in _forms() if f[0] == form)
    opt = RendererCpuOption(diffuse_color=DiffuseColor.kVertex, backface_culling=culling)
    r = Raytracer(opt)
    r.set_mesh(mesh)
    assert r.PrepareMesh()
    rc, ref, _ = O.raytrace(mesh, O.camera_from_abi(cam.to_abi()), opt, c2w_t=cam.c2w[:3, 3])
    assert rc == 0
    for _ in range(2):  # the second call starts with the bins the first one left
        out = r.render_batch([cam])[0]
        for k in ("face_id", "mask", "color"):
            assert np.array_equal(out[k], ref[k]), (form, k)
        for k in ("depth", "normal"):
            np.testing.assert_allclose(out[k], ref[k], rtol=1e-5, atol=1e-7)
    if form not in ("one_pixel", "far_away"):
        assert (ref["face_id"] >= 0).sum() > 5 or culling
