"""contiguous_u8 equals np.ascontiguousarray(img, np.uint8) for every order, stride
and type of the image."""
import numpy as np
import pytest

from ugu_amd.visibility import contiguous_u8


@pytest.mark.parametrize("dtype", [np.uint8, np.float32, np.int64])
@pytest.mark.parametrize("shape", [(5, 7, 3), (1, 1, 4), (6, 4, 1), (3, 2, 9), (4, 6), (0, 4, 3)])
def test_equals_numpy(shape, dtype):
    a = (np.random.default_rng(0).random(shape) * 255).astype(dtype)
    for img in (a, a[::-1], np.asfortranarray(a), a.T, a[:, ::2], a[..., ::-1], a.tolist()):
        want = np.ascontiguousarray(img, np.uint8)
        got = contiguous_u8(img)
        assert got.flags.c_contiguous and got.dtype == np.uint8 and got.shape == want.shape
        assert np.array_equal(got, want)
