"""Copies to and from pageable arrays at the sizes where their paths change: the plain
copy below 4 KB out of and 64 KB into the device, one chunk (32 KB), the host threads
(512 KB), one group of 128 chunks (4 MB), the ring of two groups (8 MB) and its reuse.
Out of the device against the same pass's planes in device memory, into it by texture
mapping against oracle_texture_map, byte for byte."""
import threading

import numpy as np
import pytest

import oracle as O
from ugu_amd import DiffuseColor, Rasterizer, RendererCpuOption, _abi, scenes, texturing

pytestmark = pytest.mark.gpu


def _renderer():
    m = scenes.perturbed_sphere(*scenes.icosphere_unit(3))
    m.set_vertex_colors(np.random.default_rng(0).random((len(m.vertices), 3), np.float32) * 255)
    r = Rasterizer(RendererCpuOption(diffuse_color=DiffuseColor.kVertex))
    r.set_mesh(m)
    assert r.PrepareMesh()
    return r


def _camera(w, h):
    return scenes.ring_cameras(1, 3.0, 1, 0, res_choices=[(w, h)])[0]


KINDS = {"depth": ((), "float32"), "face_id": ((), "int32"), "mask": ((), "uint8"),
         "normal": ((3,), "float32"), "color": ((3,), "uint8")}


def _device(r, cam, names):
    import torch
    bufs = {k: torch.full((cam.height, cam.width) + KINDS[k][0], 77,
                          dtype=getattr(torch, KINDS[k][1]), device="cuda") for k in names}
    torch.cuda.synchronize()
    r.render_device([cam], [bufs])
    return {k: t.cpu().numpy() for k, t in bufs.items()}


def _equal(host, dev, label):
    for k in dev:
        assert host[k].reshape(dev[k].shape).tobytes() == dev[k].tobytes(), (label, k)


# pixels of a 4-byte plane: 4 KB, 32 KB, 512 KB, 4 MB and 8 MB, each a pixel or a few
# below, at and above; three groups; and one pixel
SIZES = [(33, 31), (32, 32), (41, 25), (8191, 1), (128, 64), (8193, 1), (255, 514), (512, 256),
         (12, 10923), (1023, 1025), (1024, 1024), (460, 2279), (6223, 337), (2048, 1024),
         (387, 5419), (2048, 1537), (1, 1)]


@pytest.mark.parametrize("w,h", SIZES)
def test_out_of_the_device(gpu_available, w, h):
    r, cam = _renderer(), _camera(w, h)
    for names in (("depth",), ("color", "depth", "normal", "mask", "face_id")):
        dev = _device(r, cam, names)
        for call in range(2):
            _equal(r.render_batch([cam], outputs=names)[0], dev, (names, call))


WIDTH = 8192


def _rows(sizes, seed):
    """Images of one row of sizes[k] pixels, and faces that sample image k over its whole
    length into row k of a texture: every chunk of the images is read, a dozen times at
    the least."""
    rng = np.random.default_rng(seed)
    images = [rng.integers(0, 256, (1, s, 3), dtype=np.uint8) for s in sizes]
    n = len(sizes)
    recs, orecs = (_abi.UguTexFace * n)(), (O.OracleTexFace * n)()
    for k, s in enumerate(sizes):
        for r in (recs[k], orecs[k]):
            r.keyframe = k
            for q, (src, dst) in enumerate(zip((0, 0, 2 * s, 0, 0, 2),
                                               (0, k, 2 * WIDTH, k, 0, k + 2))):
                r.src[q], r.dst[q] = float(src), float(dst)
    return images, recs, orecs, n


# bytes of all images: 64 KB with its records and descriptors (52 and 16 bytes an
# image), 512 KB, 4 MB, 8 MB, 12 MB and 20 MB, a few bytes below, at and above
BYTES = [3, 32766, 32769, 65331, 65334, 65466, 65469, 65535, 524286, 524289, 4194303, 4194306,
         8388606, 8388609, 12582912, 12582915, 20971521]


@pytest.mark.parametrize("total", BYTES)
@pytest.mark.parametrize("parts", [1, 3])
def test_into_the_device(gpu_available, total, parts):
    px = total // 3
    sizes = [px] if parts == 1 else [max(1, px // 7), max(1, px // 2), max(1, px - px // 7 - px // 2)]
    images, recs, orecs, n = _rows(sizes, total)
    want = O.texture_map(images, orecs, WIDTH, n, 0)
    for _ in range(2):
        got = texturing.texture_map_faces(images, recs, n, WIDTH, n, 0)
        for a, b in zip(got, want):
            assert np.array_equal(a, b)


def test_threads_reuse_their_rings(gpu_available):
    """Four threads at once, 20 MB into and 8 MB out of the device, and passes whose
    planes take the ring three times."""
    jobs = [_rows([2_333_333 + 1000 * k, 1_700_000, 2_900_001], k) for k in range(2)]
    want = [O.texture_map(j[0], j[2], WIDTH, j[3], 0) for j in jobs]
    rs, cam = [_renderer() for _ in range(2)], _camera(1600, 1000)
    dev = _device(rs[0], cam, tuple(KINDS))
    bad = []

    def guarded(fn, *args):
        try:
            for _ in range(4):
                fn(*args)
        except BaseException as e:  # noqa: BLE001 - reported by the caller
            bad.append(e)

    def upload(k):
        images, recs, _, n = jobs[k]
        for a, b in zip(texturing.texture_map_faces(images, recs, n, WIDTH, n, 0), want[k]):
            assert np.array_equal(a, b)

    def render(r):
        _equal(r.render_batch([cam], outputs=tuple(KINDS))[0], dev, "thread")

    ts = [threading.Thread(target=guarded, args=(upload, k)) for k in range(2)] + \
         [threading.Thread(target=guarded, args=(render, r)) for r in rs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad
