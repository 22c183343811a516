"""Outputs in host memory come through pinned slots of 1 MB that host threads
empty; they must equal, byte for byte, the same pass's outputs in device memory,
at plane sizes around the slot size and around the total (512 KB) below which one
plain copy is made, with several planes per pass and from several threads."""
import threading

import numpy as np
import pytest

from ugu_amd import DiffuseColor, Rasterizer, Raytracer, RendererCpuOption, scenes

pytestmark = pytest.mark.gpu

# 4-byte planes: just below 512 KB, 512 KB, just below 1 MB, 1 MB, just above 1 MB,
# 9 MB (more chunks than slots), 9 KB
SIZES = [(4369, 30), (512, 256), (4095, 64), (512, 512), (2731, 96), (1536, 1536), (61, 37)]


def _renderer(cls):
    v, f = scenes.icosphere_unit(3)
    m = scenes.perturbed_sphere(v, f)
    m.set_vertex_colors(np.random.default_rng(0).random((len(m.vertices), 3), np.float32) * 255)
    r = cls(RendererCpuOption(diffuse_color=DiffuseColor.kVertex))
    r.set_mesh(m)
    assert r.PrepareMesh()
    return r


def _device(r, cams, names):
    import torch
    kinds = {"depth": ((), torch.float32), "face_id": ((), torch.int32),
             "mask": ((), torch.uint8), "normal": ((3,), torch.float32),
             "color": ((3,), torch.uint8)}
    bufs = [{k: torch.full((c.height, c.width) + kinds[k][0], 77, dtype=kinds[k][1],
                           device="cuda") for k in names} for c in cams]
    torch.cuda.synchronize()
    r.render_device(cams, bufs)
    return [{k: t.cpu().numpy() for k, t in b.items()} for b in bufs]


def _equal(host, dev, label):
    for h, d in zip(host, dev):
        for k in d:
            assert h[k].reshape(d[k].shape).tobytes() == d[k].tobytes(), (label, k)


@pytest.mark.parametrize("names", [("depth",), ("color", "depth", "normal", "mask", "face_id")])
@pytest.mark.parametrize("cls", [Rasterizer, Raytracer])
def test_planes_equal_device(gpu_available, cls, names):
    r = _renderer(cls)
    cams = [scenes.ring_cameras(1, 3.0, 3 + k, 0, res_choices=[s])[0]
            for k, s in enumerate(SIZES)]
    for c in cams:
        _equal(r.render_batch([c], outputs=names), _device(r, [c], names), (c.width, c.height))
    _equal(r.render_batch(cams, outputs=names), _device(r, cams, names), "all")


def test_threads(gpu_available):
    cam = scenes.ring_cameras(1, 3.0, 5, 0, res_choices=[(1200, 900)])[0]
    names = ("color", "depth", "normal", "mask", "face_id")
    rs = [_renderer(Rasterizer) for _ in range(4)]
    want = _device(rs[0], [cam], names)
    bad = []

    def work(r):
        try:
            for _ in range(10):
                _equal(r.render_batch([cam], outputs=names), want, "thread")
        except BaseException as e:  # noqa: BLE001 - reported by the caller
            bad.append(e)

    ts = [threading.Thread(target=work, args=(r,)) for r in rs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad


def test_texture_map_calls_share_nothing(gpu_available):
    """texture_map_faces keeps one idle context: calls of changing sizes, after an
    error and from several threads give what a first call gives."""
    from ugu_amd import _abi, texturing

    def job(seed):
        rng = np.random.default_rng(seed)
        n, tex = int(rng.integers(1, 400)), int(rng.integers(16, 700))
        images = [(rng.random((int(rng.integers(8, 500)), 300, 3)) * 255).astype(np.uint8)
                  for _ in range(int(rng.integers(1, 5)))]
        recs = (_abi.UguTexFace * n)()
        for r in recs:
            r.keyframe = int(rng.integers(-1, len(images)))
            for k in range(6):
                r.src[k] = float(rng.uniform(0, 299))
                r.dst[k] = float(rng.uniform(-2, tex + 2))
        return images, recs, n, tex, tex, 3

    def fresh(j):
        texturing._release_spares()
        return texturing.texture_map_faces(*j)

    jobs = [job(s) for s in range(8)]
    want = [fresh(j) for j in jobs]
    bad = []

    def work(first):
        try:
            for k in range(16):
                i = (first + k) % len(jobs)
                for a, b in zip(texturing.texture_map_faces(*jobs[i]), want[i]):
                    assert np.array_equal(a, b), i
                with pytest.raises(_abi.HipError):
                    texturing.texture_map_faces(*jobs[i][:3], 0, 16, 3)
        except BaseException as e:  # noqa: BLE001 - reported by the caller
            bad.append(e)

    work(0)
    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
    assert len(texturing._spare) <= 1
