"""Passes of one context after each other: a pass of one view starts with the
tile counters the passes before it left, so every order of one view and many,
of view sizes, tile shapes, overflowing bins, rasterizer and raytracer passes has
to give what a fresh context gives, bit for bit."""
import numpy as np
import pytest

from ugu_amd import DiffuseColor, Rasterizer, Raytracer, RendererCpuOption, scenes

pytestmark = pytest.mark.gpu

SIZES = [(160, 120), (33, 17), (257, 190), (16, 16)]


def _mesh():
    v, f = scenes.icosphere_unit(4)
    m = scenes.perturbed_sphere(v, f)
    m.set_vertex_colors(np.random.default_rng(0).random((len(m.vertices), 3), np.float32) * 255)
    return m


def _renderer(cls, mesh):
    r = cls(RendererCpuOption(diffuse_color=DiffuseColor.kVertex))
    r.set_mesh(mesh)
    assert r.PrepareMesh()
    return r


@pytest.mark.parametrize("cls", [Rasterizer, Raytracer])
@pytest.mark.parametrize("seed", range(4))
def test_sequences(gpu_available, cls, seed):
    mesh = _mesh()
    rng = np.random.default_rng(seed)
    cams = [scenes.ring_cameras(2, 3.0, 3 + k, 0, res_choices=[s])[0]
            for k, s in enumerate(SIZES)]
    fresh = [_renderer(cls, mesh).render_batch([c])[0] for c in cams]
    r = _renderer(cls, mesh)
    for _ in range(25):
        n = int(rng.choice([1, 1, 1, 2, 3, 13]))  # 13: more views than kernel arguments hold
        pick = rng.integers(0, len(cams), n)
        if cls is Rasterizer and rng.random() < 0.4:
            tile = [(8, 8), (16, 16), (32, 8)][rng.integers(0, 3)]
            r.set_tiling(*tile, bin_capacity=int(rng.choice([8, 1024])),
                         persistent=bool(rng.random() < 0.5))
        out = r.render_batch([cams[i] for i in pick])
        for i, o in zip(pick, out):
            for k in o:
                assert np.array_equal(o[k], fresh[i][k]), (n, SIZES[i], k)
