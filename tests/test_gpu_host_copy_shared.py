"""Views of one call that are given the same host arrays, wholly or in part: the
planes are copied in the order of the views, so the last view's bytes stay."""
import numpy as np
import pytest

from ugu_amd import DiffuseColor, Rasterizer, Raytracer, RendererCpuOption, _abi, scenes
from ugu_amd.renderer import options_to_abi

pytestmark = pytest.mark.gpu

OPTION = RendererCpuOption(diffuse_color=DiffuseColor.kVertex)


def _call(r, name, cams, arrays):
    """Renders the depth planes of the views into `arrays` (one address per view)."""
    outs = (_abi.UguOutputs * len(cams))()
    for o, a in zip(outs, arrays):
        o.depth = a
    abi = (_abi.UguCamera * len(cams))(*[c.to_abi() for c in cams])
    rc = getattr(r._lib, name)(r._ctx, abi, len(cams), options_to_abi(OPTION), outs,
                               _abi.UGU_HIP_MEMORY_HOST)
    assert rc == 0, r._lib.ugu_hip_last_error(r._ctx)


# planes of one 32 KB chunk, of two, of 1.2 MB; 600 KB to 40 MB in all
@pytest.mark.parametrize("w,h,n", [(104, 78, 24), (128, 96, 20), (640, 480, 32)])
@pytest.mark.parametrize("shift", [0, 4096])
@pytest.mark.parametrize("cls,name", [(Rasterizer, "ugu_hip_render_batch"),
                                      (Raytracer, "ugu_hip_raytrace")])
def test_last_view_stays(gpu_available, w, h, n, shift, cls, name):
    m = scenes.perturbed_sphere(*scenes.icosphere_unit(3))
    m.set_vertex_colors(np.random.default_rng(0).random((len(m.vertices), 3), np.float32) * 255)
    r = cls(OPTION)
    r.set_mesh(m)
    assert r.PrepareMesh()
    cams = scenes.ring_cameras(n, 3.0, 2, 0, res_choices=[(w, h)])
    size = w * h * 4
    views = np.zeros((n, size), np.uint8)
    _call(r, name, cams, [v.ctypes.data for v in views])
    want = np.zeros(size + shift * (n - 1), np.uint8)
    for k, v in enumerate(views):
        want[shift * k:shift * k + size] = v
    for _ in range(20):
        got = np.zeros_like(want)
        _call(r, name, cams, [got.ctypes.data + shift * k for k in range(n)])
        assert np.array_equal(got, want)
