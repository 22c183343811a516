"""Faces over many of a view's tiles: the raytracer keeps them in a list per view
that every tile goes through. Faces at the limit of 16 tiles, more of them than a
list holds, several views, and lists left by other calls; against oracle_raytrace,
every output exactly but depth and normal (1e-5 relative, as in the raytracer's other
parity tests)."""
import numpy as np
import pytest

import oracle as O
from ugu_amd import DiffuseColor, Mesh, PinholeCamera, Raytracer, RendererCpuOption, scenes

pytestmark = pytest.mark.gpu

TILE = 16
OPTION = RendererCpuOption(diffuse_color=DiffuseColor.kVertex)


def _mesh(tris, seed=0):
    v = np.asarray(tris, np.float32).reshape(-1, 3)
    m = Mesh(v, np.arange(len(v), dtype=np.int32))
    m.CalcFaceNormal()
    m.set_normals(np.repeat(m.face_normals, 3, axis=0))
    m.set_normal_indices(m.vertex_indices)
    m.set_vertex_colors(np.random.default_rng(seed).random((len(v), 3), np.float32) * 255)
    return m


def _camera(w, h, dx=0.0, f=None):
    c2w = np.eye(4)
    c2w[0, 3] = dx
    f = f or 0.9 * h
    return PinholeCamera(w, h, c2w, (w * 0.5 - 0.5, h * 0.5 - 0.5), (f, f))


def _boxes(cam, n, tiles, seed):
    """n triangles whose boxes span tiles[k] x tiles[k] tiles of the view, at random
    places and depths, of either winding."""
    rng = np.random.default_rng(seed)
    c, f = np.asarray(cam.principal_point), np.asarray(cam.focal_length)
    out = []
    for k in range(n):
        s = TILE * tiles[k % len(tiles)] - 3.0
        at = TILE * rng.integers(0, [max(1, cam.width // TILE - 2), max(1, cam.height // TILE - 2)]) + 1.0
        # thin, along a diagonal: most of them are seen somewhere
        xy = at + np.array([[0.0, 0.1], [s, s], [rng.uniform(0.0, 0.1) * s, 1.5]])
        z = rng.uniform(2.0, 20.0) + rng.uniform(-0.5, 0.5, (3, 1))
        p = np.concatenate([(xy - c) / f * z, z], 1)
        out.append(p[::-1] if rng.random() < 0.5 else p)
    return np.asarray(out)


def _reference(mesh, cam):
    rc, ref, _ = O.raytrace(mesh, O.camera_from_abi(cam.to_abi()), OPTION, c2w_t=cam.c2w[:3, 3])
    assert rc == 0
    return ref


def _check(out, ref, label):
    for k in ("face_id", "mask", "color"):
        assert np.array_equal(out[k], ref[k]), (label, k)
    for k in ("depth", "normal"):
        np.testing.assert_allclose(out[k], ref[k], rtol=1e-5, atol=1e-7)


def _renderer(mesh):
    r = Raytracer(OPTION)
    r.set_mesh(mesh)
    assert r.PrepareMesh()
    return r


# 4 x 4 tiles stay in the bins, 5 x 4 and more go to the list
@pytest.mark.parametrize("tiles", [(4,), (5,), (1, 4, 5, 9)])
@pytest.mark.parametrize("n", [70, 600])
def test_at_the_limit(gpu_available, tiles, n):
    cam = _camera(333, 241)
    mesh = _mesh(_boxes(cam, n, tiles, n))
    ref = _reference(mesh, cam)
    r = _renderer(mesh)
    for call in range(3):
        _check(r.render_batch([cam])[0], ref, call)


def test_more_than_a_list_holds(gpu_available):
    cam = _camera(200, 120)
    mesh = _mesh(_boxes(cam, 4096 + 300, (5, 6, 7), 1))
    ref = _reference(mesh, cam)
    r = _renderer(mesh)
    for call in range(3):
        _check(r.render_batch([cam])[0], ref, call)


def test_views_take_turns(gpu_available):
    """Each view has its own list; calls of other views, counts and sizes, with a
    rasterizer pass of the same renderer between them, find clear counters."""
    cams = [_camera(180 + 16 * (k % 3), 130 + 9 * (k % 4), 0.1 * k) for k in range(14)]
    mesh = _mesh(np.concatenate([_boxes(cams[0], 90, (6, 7, 1), 3),
                                 _boxes(cams[5], 60, (1,), 4)]))
    refs = [_reference(mesh, c) for c in cams]
    r = _renderer(mesh)
    for first, n in ((0, 1), (0, 3), (3, 1), (3, 1), (0, 14), (4, 2), (5, 1), (0, 13), (6, 1)):
        for k, out in enumerate(r.render_batch(cams[first:first + n])):
            _check(out, refs[first + k], (first, n, k))


def test_faces_around_the_camera(gpu_available):
    """Faces without a bound (across the camera's plane) cover the whole view."""
    rng = np.random.default_rng(2)
    tris = rng.uniform(-2, 2, (300, 1, 3)) + rng.uniform(-2.5, 2.5, (300, 3, 3))
    cam = _camera(97, 71)
    mesh = _mesh(tris)
    _check(_renderer(mesh).render_batch([cam])[0], _reference(mesh, cam), "around")


def test_large_faces_do_not_serialize_the_setup(gpu_available):
    """A ball in a room of 12 triangles at 1920 x 1080: with the room's faces appended
    to 2 x 8160 bins by two wavefronts the pass took 20 times the ball's alone."""
    ball = scenes.perturbed_sphere(*scenes.icosphere_unit(5))
    v = np.asarray(ball.vertices)[np.asarray(ball.vertex_indices).reshape(-1, 3)] * 0.5 + [0, 0, 3.0]
    s, quads = 5.0, []
    for axis in range(3):
        for side in (-s, s):
            q = np.zeros((4, 3))
            q[:, axis] = side
            q[:, (axis + 1) % 3] = [-s, s, s, -s]
            q[:, (axis + 2) % 3] = [-s, -s, s, s]
            quads += [q[[0, 1, 2]], q[[0, 2, 3]]]

    def gpu_ms(tris):
        import torch
        r = _renderer(_mesh(tris))
        r.enable_profiling()
        buf = {"face_id": torch.zeros((1080, 1920), dtype=torch.int32, device="cuda")}
        torch.cuda.synchronize()
        ms = []
        for _ in range(7):
            r.render_device([_camera(1920, 1080)], [buf])
            ms.append(r.timings()["raster_ms"])
        return np.median(ms[1:])

    alone = gpu_ms(v)
    room = gpu_ms(np.concatenate([v, np.asarray(quads)]))
    assert room < 4.0 * alone, (room, alone)


def test_share_of_the_tiles(gpu_available):
    """In a view of 16641 tiles the list takes faces over more than 32 of them."""
    small = _camera(333, 241, f=220.0)
    mesh = _mesh(_boxes(small, 400, (4, 5, 6, 9), 8))
    ref = _reference(mesh, small)
    at = 16 * 50
    c = np.asarray(small.principal_point) + at
    cam = PinholeCamera(2064, 2064, np.eye(4), tuple(c), tuple(small.focal_length))
    r = _renderer(mesh)
    for call in range(2):
        out = r.render_batch([cam])[0]
        _check({k: v[at:at + 241, at:at + 333] for k, v in out.items()}, ref, call)


@pytest.mark.parametrize("views", [1, 5, 40])
def test_few_faces_many_views(gpu_available, views):
    """Blocks of the setup take one view each where they are few."""
    cams = [_camera(64 + k % 5, 48, 0.02 * k) for k in range(views)]
    mesh = _mesh(_boxes(cams[0], 50, (1, 2), 9))
    r = _renderer(mesh)
    for k, out in enumerate(r.render_batch(cams)):
        _check(out, _reference(mesh, cams[k]), k)
