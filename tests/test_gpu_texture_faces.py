"""Texture mapping against oracle_texture_map, bit for bit, where its kernels can go
wrong: boxes of one texel up to the whole texture, faces outside the texture, without
a keyframe, without area or not finite, no face at all, and textures whose number of
texels is around the 256 of a block."""
import numpy as np
import pytest

import oracle as O
from ugu_amd import texturing as T

pytestmark = pytest.mark.gpu

W, H = 301, 173
SIZES = [(0.2, 0.2), (13.9, 13.9), (14.9, 13.9), (253.9, -0.1), (254.9, -0.1), (0.5, 160.0),
         (300.0, 172.0), (3.0, 4.0), (30.0, 40.0)]


def _faces(n, rng):
    out = []
    for i in range(n):
        w, h = SIZES[rng.integers(0, len(SIZES))]
        x, y = rng.uniform(-3, W), rng.uniform(-3, H)
        if w > 200:
            x = 0.0
        if h > 100:
            y = 0.0
        d = np.array([[x, y], [x + w, y + h * rng.random()], [x + w * rng.random(), y + h]])
        kind = rng.integers(0, 12)
        if kind == 0:
            d[2] = d[1]
        if kind == 1:
            d[rng.integers(0, 3), rng.integers(0, 2)] = rng.choice([np.nan, np.inf, -np.inf, 3e9])
        if kind == 2:
            d += 1000
        out.append((int(rng.integers(-1, 3)), rng.uniform(1, 58, 6), d.reshape(-1)))
    return out


@pytest.mark.parametrize("tw, th", [(W, H), (16, 16), (255, 1), (1, 257), (1, 1)])
@pytest.mark.parametrize("n", [0, 1, 5, 64, 400])
def test_boxes_match_oracle(gpu_available, n, tw, th):
    rng = np.random.default_rng(n)
    imgs = [rng.integers(0, 256, (60, 60 + k, 3), dtype=np.uint8) for k in range(3)]
    faces = _faces(n, rng)
    recs, orecs = (T._abi.UguTexFace * max(1, n))(), (O.OracleTexFace * n)()
    for i, (kf, src, dst) in enumerate(faces):
        for r in (recs[i], orecs[i]):
            r.keyframe = kf
            for k in range(6):
                r.src[k] = float(np.float32(src[k]))
                r.dst[k] = float(np.float32(dst[k]))
    for pad in (0, 3):
        tex, mask = T.texture_map_faces(imgs, recs, n, tw, th, pad)
        rt, rm = O.texture_map(imgs, orecs, tw, th, pad)
        assert np.array_equal(mask, rm)
        assert np.array_equal(tex, rt)
