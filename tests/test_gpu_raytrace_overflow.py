"""Passes of the raytracer in which a tile's bin overflows only when its front and
back faces are taken together: each segment fits the bin's first 1024 entries, so
the setup kernel sees no overflow and the tile kernel finds it, in some tiles,
while the others work. Against oracle_raytrace, every output exactly but depth and
normal (within 1e-5 relative, as the raytracer's other parity tests)."""
import numpy as np
import pytest

import oracle as O
from ugu_amd import DiffuseColor, Mesh, PinholeCamera, Raytracer, RendererCpuOption

pytestmark = pytest.mark.gpu

TILE = 16


def _clusters(w, h, full, per_side, others, seed, far=5.0):
    """Triangles three pixels wide, whole inside one tile each: `per_side` clockwise
    and as many counter-clockwise ones on screen in every tile of `full`, `others`
    of each in every other tile."""
    rng = np.random.default_rng(seed)
    tx, ty = -(-w // TILE), -(-h // TILE)
    f = 0.9 * h
    c = np.array([w * 0.5 - 0.5, h * 0.5 - 0.5])
    shape = np.array([[-1.5, -1.2], [1.5, -1.0], [0.2, 1.6]])
    pts = []
    for t in range(tx * ty):
        n = per_side if t in full else others
        lo = np.array([t % tx, t // tx]) * TILE + 2.0
        for flip in (False, True):
            at = lo + rng.uniform(0.0, TILE - 5.0, (n, 1, 2))
            xy = at + (shape[::-1] if flip else shape)
            z = rng.uniform(2.0, far, (n, 1, 1)).repeat(3, 1)
            pts.append(np.concatenate([(xy - c) / f * z, z], -1))
    p = np.concatenate(pts)
    p = p[rng.permutation(len(p))]
    m = Mesh(p.reshape(-1, 3).astype(np.float32), np.arange(p.shape[0] * 3, dtype=np.int32))
    m.CalcFaceNormal()
    m.set_normals(np.repeat(m.face_normals, 3, axis=0))
    m.set_normal_indices(m.vertex_indices)
    m.set_vertex_colors(rng.random((len(m.vertices), 3), np.float32) * 255)
    return m, PinholeCamera(w, h, np.eye(4), tuple(c), (f, f))


def _check(out, ref, label):
    for k in ("face_id", "mask", "color"):
        assert np.array_equal(out[k], ref[k]), (label, k)
    for k in ("depth", "normal"):
        np.testing.assert_allclose(out[k], ref[k], rtol=1e-5, atol=1e-7)


AT = 960  # where the small view lies in the large one, in x and y


def _large(cam):
    """A view with the small one at (AT, AT), of so many tiles (16641) that the bins
    start with 1024 entries each; fewer tiles get more of the same memory."""
    c = np.asarray(cam.principal_point) + AT
    return PinholeCamera(2064, 2064, np.eye(4), tuple(c), tuple(cam.focal_length))


def _crop(out, w, h):
    mask = out["mask"].copy()
    mask[AT:AT + h, AT:AT + w] = 0
    assert not mask.any()
    return {k: v[AT:AT + h, AT:AT + w] for k, v in out.items()}


@pytest.mark.parametrize("full", [(0,), (3, 17, 29, 59), tuple(range(0, 60, 6))])
@pytest.mark.parametrize("views", [1, 2])
def test_segments_overflow_together(gpu_available, full, views):
    mesh, cam = _clusters(160, 96, full, 700, 20, len(full))
    opt = RendererCpuOption(diffuse_color=DiffuseColor.kVertex)
    rc, ref, _ = O.raytrace(mesh, O.camera_from_abi(cam.to_abi()), opt, c2w_t=cam.c2w[:3, 3])
    assert rc == 0 and (ref["face_id"] >= 0).sum() > 1000
    r = Raytracer(opt)
    r.set_mesh(mesh)
    assert r.PrepareMesh()
    for call in range(2):
        for out in r.render_batch([_large(cam)] * views):
            _check(_crop(out, 160, 96), ref, call)
        assert r.timings()["retries"] == 1 - call
    for out in r.render_batch([cam] * views):
        _check(out, ref, "small")


def _retries(r, cam, calls):
    """Repeated passes of each of `calls` calls, whose outputs are all equal."""
    out, first = [], None
    for _ in range(calls):
        got = r.render_batch([cam], outputs=("face_id", "depth"))[0]
        out.append(r.timings()["retries"])
        first = first or got
        for k in got:
            assert np.array_equal(got[k], first[k])
    return out


def test_dense_tile_is_not_tried_on_every_call(gpu_available):
    """2500 front and 2500 back faces on a tile exceed what a bin may hold (4096): the
    hierarchy traces the view, and the bins are tried again ever more rarely. After
    PrepareMesh, and for a view of other tiles, they are tried at once."""
    mesh, cam = _clusters(160, 96, (17,), 2500, 20, 3, far=9.0)  # few layers from the side
    corner = PinholeCamera(64, 48, np.eye(4), tuple(cam.principal_point), tuple(cam.focal_length))
    r = Raytracer(RendererCpuOption(diffuse_color=DiffuseColor.kVertex))
    r.set_mesh(mesh)
    for _ in range(2):
        assert r.PrepareMesh()
        tried = [k for k, n in enumerate(_retries(r, cam, 300)) if n > 0]
        assert tried == [0, 2, 6, 14, 30, 62, 126, 254]
    assert _retries(r, corner, 2) == [0, 0]  # its tiles hold few faces


def test_bins_that_grew_are_kept(gpu_available):
    mesh, cam = _clusters(160, 96, (17,), 1500, 20, 4)
    r = Raytracer(RendererCpuOption(diffuse_color=DiffuseColor.kVertex))
    r.set_mesh(mesh)
    assert r.PrepareMesh()
    assert _retries(r, _large(cam), 4) == [1, 0, 0, 0]
    assert _retries(r, cam, 2) == [0, 0]


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
def test_faces_that_are_not_finite_fill_no_bins(gpu_available, value):
    """5000 faces with such a coordinate can be hit nowhere. Put into every tile's bin
    they would exceed it and send each call to the hierarchy."""
    mesh, cam = _clusters(160, 96, (17,), 100, 20, 5)
    rng = np.random.default_rng(6)
    more = rng.uniform(-1, 1, (15000, 3)).astype(np.float32)
    more[np.arange(0, 15000, 3) + rng.integers(0, 3, 5000), rng.integers(0, 3, 5000)] = value
    v = np.concatenate([more, mesh.vertices])
    m = Mesh(v, np.arange(len(v), dtype=np.int32))
    m.set_face_normals(np.concatenate([np.tile(np.float32([0, 0, 1]), (5000, 1)),
                                       mesh.face_normals]))
    m.set_normals(np.tile(np.float32([0, 0, -1]), (len(v), 1)))
    m.set_normal_indices(m.vertex_indices)
    m.set_vertex_colors(rng.random((len(v), 3), np.float32) * 255)
    opt = RendererCpuOption(diffuse_color=DiffuseColor.kVertex)
    rc, ref, _ = O.raytrace(m, O.camera_from_abi(cam.to_abi()), opt, c2w_t=cam.c2w[:3, 3])
    assert rc == 0 and (ref["face_id"] >= 5000).sum() > 1000
    r = Raytracer(opt)
    r.set_mesh(m)
    assert r.PrepareMesh()
    for call in range(2):
        _check(r.render_batch([cam])[0], ref, value)
        assert r.timings()["retries"] == 0


def _used():
    import torch
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def _masks(r, cams):
    import torch
    bufs = [{"mask": torch.zeros((c.height, c.width), dtype=torch.uint8, device="cuda")}
            for c in cams]
    torch.cuda.synchronize()
    r.render_device(cams, bufs)
    return [b["mask"] for b in bufs]


def test_memory_of_the_bins(gpu_available):
    """A dense tile of one mesh does not size the bins of the next mesh's views (262144
    tiles: 2 GiB for 1024 faces each, 7 GiB for what the first mesh needed), and views
    whose bins would take more than 8 GiB go to the hierarchy."""
    import torch
    r = Raytracer(RendererCpuOption(diffuse_color=DiffuseColor.kVertex))
    dense, cam = _clusters(160, 96, (17,), 1500, 20, 4)
    r.set_mesh(dense)
    assert r.PrepareMesh()
    _retries(r, cam, 2)
    ball, _ = _clusters(160, 96, (17,), 100, 20, 5)
    r.set_mesh(ball)
    assert r.PrepareMesh()
    cams = [PinholeCamera(2048, 2048, np.eye(4), (1023.5 - k, 1000.0), (1800.0, 1800.0))
            for k in range(80)]
    one = _masks(r, cams[:1])[0].cpu()
    before = _used()
    few = _masks(r, cams[:16])
    assert _used() - before < 3 << 30
    assert torch.equal(few[0].cpu(), one) and bool(one.any())
    held = _used()
    many = _masks(r, cams)
    assert _used() - held < 1 << 30
    for a, b in zip(few, many):
        assert torch.equal(a, b)
