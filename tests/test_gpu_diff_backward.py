"""The backward pass's kernels at the sizes where they branch, against the
float64 CPU backward: every set of learned parameters (each its own kernel),
more views than cameras kept in LDS, faces of many pixels (sums by scans), of
about one and of less, textures larger than a block's table, one texel, one
pixel, sizes that are no multiple of a tile. Gradients are float32 sums of
float64 terms; n terms of one sign carry at most n 2^-24 relative error, and no
vertex or texel here gets more than a few hundred block sums, so 2e-5 norm-wise
holds with a margin; a missed or doubled term is far above it."""
import numpy as np
import pytest

import oracle as O
from ugu_amd import scenes

pytestmark = pytest.mark.gpu

TOL = 2e-5


def _mesh(level):
    v, f = scenes.icosphere_unit(level)
    return scenes.perturbed_sphere(v, f)


def _check(mesh, cams, learn, tex_size, repeat=1):
    import torch
    from ugu_amd.diff import DiffRenderer
    rng = np.random.default_rng(len(cams) * 131 + tex_size)
    colors = rng.random((len(mesh.vertices), 3), np.float32) if "c" in learn or not tex_size else None
    tex = rng.random((tex_size, tex_size, 3), np.float32) if tex_size else None
    dr = DiffRenderer(mesh)
    p = {"v": torch.tensor(mesh.vertices, device="cuda"),
         "c": None if colors is None else torch.tensor(colors, device="cuda"),
         "t": None if tex is None else torch.tensor(tex, device="cuda")}
    for k in learn:
        p[k].requires_grad_(True)
    for _ in range(repeat):
        img, fid = dr.render_flat(cams, p["v"], p["c"], p["t"])
        g = rng.normal(size=img.shape[0]).astype(np.float32)
        got = torch.autograd.grad(img, [p[k] for k in learn], torch.tensor(g, device="cuda"))
        want = {k: 0.0 for k in "vct"}
        at = 0
        for c in cams:
            n = c.width * c.height
            gv, gc, gt = O.diff_backward_f64(
                O.camera_from_abi(c.to_abi()), mesh, mesh.vertices, colors, tex,
                fid[at:at + n].cpu().numpy().reshape(c.height, c.width),
                g[at * 3:(at + n) * 3].reshape(c.height, c.width, 3).astype(np.float64))
            for k, x in zip("vct", (gv, gc, gt)):
                want[k] = want[k] + x if x is not None else want[k]
            at += n
        for k, x in zip(learn, got):
            x = x.cpu().numpy().astype(np.float64)
            rel = np.linalg.norm(x - want[k]) / max(np.linalg.norm(want[k]), 1e-30)
            assert rel < TOL, (k, rel)


@pytest.mark.parametrize("learn,tex_size", [("v", 0), ("c", 0), ("vc", 0), ("t", 64), ("vt", 64),
                                            ("ct", 64), ("vct", 64), ("vct", 1), ("t", 1000),
                                            ("vct", 1000)])
@pytest.mark.parametrize("level,size", [(1, (130, 97)), (4, (128, 128)), (6, (75, 61))])
def test_parameters(gpu_available, learn, tex_size, level, size):
    cams = scenes.ring_cameras(3, 3.0, 5, 6, res_choices=[size])
    _check(_mesh(level), cams, learn, tex_size)


@pytest.mark.parametrize("views", [1, 64, 65])
def test_many_views(gpu_available, views):
    cams = scenes.ring_cameras(views, 3.0, 7, 8, res_choices=[(33, 17), (48, 40)])
    _check(_mesh(3), cams, "vct", 40, repeat=2)


def test_one_pixel(gpu_available):
    cams = scenes.ring_cameras(2, 1.5, 9, 10, res_choices=[(1, 1)])
    _check(_mesh(2), cams, "vct", 8)


def test_large_pass(gpu_available):
    """Several items per thread, and blocks whose vertices and texels exceed
    the tables. No view lies in the mesh's plane of symmetry: there a pixel
    column falls on the uv seam's edge, where the clamped texture has a kink and
    the position gradient is undefined (weights of 1e-16 of either sign)."""
    cams = scenes.ring_cameras(5, 2.2, 11, 12, res_choices=[(1283, 1021)])[1:]
    _check(_mesh(7), cams, "vct", 2048)
