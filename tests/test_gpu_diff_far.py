"""The differentiable image's weights far from the origin, against the same model in
80-bit arithmetic. A face's uvs spread over +-1e6 but come to 0.4 at one pixel, so that
a weight's error shows 4e9 times as large in the 4096 texels wide texture."""
import numpy as np
import pytest

from ugu_amd import Mesh, PinholeCamera
from ugu_amd.diff import DiffRenderer

pytestmark = pytest.mark.gpu

L = np.longdouble
W, H, F, DEPTH, TW = 640, 400, 1000.0, 3.0, 4096


def _weights(cam, verts, x, y):
    """Perspective-correct weights of the corners (n, 3, 3) at the pixels."""
    R = np.array(cam.w2c_R, dtype=np.float32).astype(L).reshape(3, 3)
    t = np.array(cam.w2c_t, dtype=np.float32).astype(L)
    q = np.einsum("ij,nkj->nki", R, verts.astype(L)) + t
    X = L(cam.fx) * q[..., 0] - (x - L(cam.cx))[:, None] * q[..., 2]
    Y = L(cam.fy) * q[..., 1] - (y - L(cam.cy))[:, None] * q[..., 2]
    a = np.stack([X[:, 2] * Y[:, 1] - X[:, 1] * Y[:, 2], X[:, 0] * Y[:, 2] - X[:, 2] * Y[:, 0],
                  X[:, 1] * Y[:, 0] - X[:, 0] * Y[:, 1]], 1)
    return a / a.sum(1, keepdims=True)


def _scene(offset, seed):
    rng = np.random.default_rng(seed)
    rot = np.linalg.qr(rng.normal(size=(3, 3)))[0]
    if np.linalg.det(rot) < 0:
        rot[:, 0] *= -1
    c2w = np.eye(4)
    c2w[:3, :3] = rot
    c2w[:3, 3] = offset * rng.normal(size=3)
    cam = PinholeCamera(W, H, c2w, (W / 2 - 0.5, H / 2 - 0.5), (F, F))
    x, y = np.meshgrid(np.arange(16, W - 16, 30), np.arange(16, H - 16, 30))
    x, y = x.reshape(-1), y.reshape(-1)
    corners = np.array([[-9.0, -7.0], [8.0, -6.0], [0.5, 9.5]]) + rng.uniform(-1, 1, (len(x), 3, 2))
    px = np.stack([x, y], 1)[:, None] + corners
    z = DEPTH + rng.uniform(-0.05, 0.05, (len(x), 3))
    q = np.stack([(px[..., 0] - (W / 2 - 0.5)) / F * z, (px[..., 1] - (H / 2 - 0.5)) / F * z, z], -1)
    verts = (np.einsum("ij,nkj->nki", rot, q) + c2w[:3, 3]).astype(np.float32)
    verts = np.concatenate([verts[:1] + 50, verts])  # face 0 is never shaded
    return cam, verts, x, y


@pytest.mark.parametrize("offset", [0.0, 30.0, 1000.0])
@pytest.mark.parametrize("seed", [0, 1])
def test_weights(gpu_available, offset, seed):
    import torch
    cam, verts, x, y = _scene(offset, seed)
    b = _weights(cam.to_abi(), verts[1:], x, y)
    rng = np.random.default_rng(seed)
    u = rng.uniform(-1e6, 1e6, (len(verts), 3)).astype(np.float32)
    u[1:, 2] = ((L(0.4) - b[:, 0] * u[1:, 0] - b[:, 1] * u[1:, 1]) / b[:, 2]).astype(np.float32)
    uv = np.stack([u, np.full_like(u, 0.25)], -1).reshape(-1, 2)
    tex = rng.random((2, TW, 3)).astype(np.float32)
    m = Mesh(verts.reshape(-1, 3), np.arange(verts.shape[0] * 3, dtype=np.int32))
    m.set_uv(uv)
    m.set_uv_indices(m.vertex_indices)
    r = DiffRenderer(m, backface_culling=False)
    image, fid = r.render_flat([cam], torch.tensor(m.vertices, device="cuda"), None,
                               torch.tensor(tex, device="cuda"))
    image = image.detach().cpu().numpy().reshape(H, W, 3)[y, x]
    fid = fid.cpu().numpy().reshape(H, W)[y, x]

    s = (b * u[1:].astype(L)).sum(1) * (TW - 1)
    at = (fid == 1 + np.arange(len(x))) & (s > 0) & (s < TW - 1)
    assert at.sum() > 100
    i = np.floor(s).astype(int).clip(0, TW - 2)
    lu = (s - i)[:, None]
    rows = [(1 - lu) * t[i] + lu * t[i + 1] for t in tex.astype(L)]
    want = 0.25 * rows[0] + 0.75 * rows[1]  # row (1 - v) (2 - 1)
    # X and Y of a corner carry 8 roundings of up to F DEPTH, the products of two corners
    # 6 of them, over a face of 15 pixels; uv of 1e6 over TW texels of contrast 1
    tol = 6 * 8 * 2.0 ** -53 * F * DEPTH / (15 * DEPTH) * 1e6 * TW + 1e-6
    assert np.abs(image - want.astype(float))[at].max() < tol
