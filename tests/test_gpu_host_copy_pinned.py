"""Host arrays in pinned memory: from 128 KB of them on the copy engine moves them
directly. Same bytes as with pageable arrays, for planes of either kind in one call,
around that limit, at odd offsets, out of the device and into it; and the first pass
into fresh pinned memory, which no CPU has touched, takes no page faults."""
import ctypes
import time

import numpy as np
import pytest

from ugu_amd import DiffuseColor, Rasterizer, RendererCpuOption, _abi, scenes
from ugu_amd.renderer import options_to_abi

pytestmark = pytest.mark.gpu

OPTION = RendererCpuOption(diffuse_color=DiffuseColor.kVertex)
BYTES = (3, 4, 12, 1, 4)  # color, depth, normal, mask, face_id


@pytest.fixture(scope="module")
def renderer(gpu_available):
    m = scenes.perturbed_sphere(*scenes.icosphere_unit(4))
    m.set_vertex_colors(np.random.default_rng(0).random((len(m.vertices), 3), np.float32) * 255)
    r = Rasterizer(OPTION)
    r.set_mesh(m)
    assert r.PrepareMesh()
    return r


def _render(r, w, h, arrays):
    cam = scenes.ring_cameras(1, 3.0, 1, 0, res_choices=[(w, h)])[0].to_abi()
    outs = _abi.UguOutputs(*[a.ctypes.data if a is not None else None for a in arrays])
    rc = r._lib.ugu_hip_render(r._ctx, ctypes.byref(cam),
                               ctypes.byref(options_to_abi(OPTION)), ctypes.byref(outs),
                               _abi.UGU_HIP_MEMORY_HOST)
    assert rc == 0, r._lib.ugu_hip_last_error(r._ctx)


def _array(n, pinned, offset=0):
    if not pinned:
        return np.full(n + offset, 77, np.uint8)[offset:]
    import torch
    return torch.full((n + offset,), 77, dtype=torch.uint8, pin_memory=True).numpy()[offset:]


# 24 bytes per pixel: below and above 128 KB of pinned planes for some of the kinds,
# 12 MB, a few pixels
@pytest.mark.parametrize("size", [(79, 69), (75, 73), (113, 97), (801, 603), (3, 2)])
@pytest.mark.parametrize("pinned", [(1, 1, 1, 1, 1), (0, 1, 0, 1, 0), (1, 0, 1, 0, 1),
                                    (0, 0, 1, 0, 0)])
def test_outputs(renderer, size, pinned):
    w, h = size
    want = [_array(b * w * h, False) for b in BYTES]
    _render(renderer, w, h, want)
    for offset in (0, 4):
        got = [_array(b * w * h, p, offset) for b, p in zip(BYTES, pinned)]
        _render(renderer, w, h, got)
        for a, b in zip(got, want):
            assert np.array_equal(a, b)


def test_first_pass_into_pinned_memory(renderer):
    """Through the slots it took four times a later pass into pageable arrays."""
    w, h = 3072, 2048
    pageable = [_array(b * w * h, False) for b in BYTES]
    later = []
    for _ in range(6):
        t = time.perf_counter()
        _render(renderer, w, h, pageable)
        later.append(time.perf_counter() - t)
    import torch
    got = [torch.empty(b * w * h, dtype=torch.uint8, pin_memory=True).numpy() for b in BYTES]
    t = time.perf_counter()
    _render(renderer, w, h, got)
    first = time.perf_counter() - t
    for a, b in zip(got, pageable):
        assert np.array_equal(a, b)
    assert first < 2.0 * np.median(later), (first, later)


@pytest.mark.parametrize("pinned", [0, 1])
@pytest.mark.parametrize("n", [1, 3])
def test_inputs(gpu_available, pinned, n):
    """Texture mapping from images, records and into planes of either kind."""
    from ugu_amd import texturing
    rng = np.random.default_rng(n)
    faces, tex = 300, 257
    images = [(rng.random((211, 300, 3)) * 255).astype(np.uint8) for _ in range(n)]
    recs = (_abi.UguTexFace * faces)()
    for r in recs:
        r.keyframe = int(rng.integers(-1, n))
        for k in range(6):
            r.src[k] = float(rng.uniform(0, 200))
            r.dst[k] = float(rng.uniform(-2, tex + 2))
    want = texturing.texture_map_faces(images, recs, faces, tex, tex, 3)
    lib = _abi.load_library()
    held, arr = [], (_abi.UguTexture * n)()
    for k, im in enumerate(images):
        a = _array(im.size, pinned if k % 2 == 0 else 0)
        a[:] = im.reshape(-1)
        held.append(a)
        arr[k] = _abi.UguTexture(im.shape[1], im.shape[0], a.ctypes.data)
    got = [_array(tex * tex * 3, pinned), _array(tex * tex, pinned)]
    ctx = lib.ugu_hip_create(0)
    try:
        for _ in range(2):
            assert lib.ugu_hip_texture_map(ctx, arr, n, recs, faces, tex, tex, 3,
                                           got[0].ctypes.data, got[1].ctypes.data) == 0
            for a, b in zip(got, want):
                assert np.array_equal(a, b.reshape(-1))
    finally:
        lib.ugu_hip_destroy(ctx)
