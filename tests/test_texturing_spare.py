"""The idle context that texture_map_faces keeps: its workspace's parts only grow, so
what counts against the limit is the largest call of each part, not the last call. The
library is replaced by a recorder; no GPU."""
import numpy as np
import pytest

from ugu_amd import _abi, texturing


class Recorder:
    def __init__(self):
        self.created, self.destroyed, self.fail = 0, [], False

    def ugu_hip_create(self, device):
        self.created += 1
        return self.created

    def ugu_hip_destroy(self, ctx):
        self.destroyed.append(ctx)

    def ugu_hip_texture_map(self, *a):
        return 1 if self.fail else 0

    def ugu_hip_last_error(self, ctx):
        return b"failed"


@pytest.fixture
def lib(monkeypatch):
    r = Recorder()
    monkeypatch.setattr(_abi, "load_library", lambda: r)
    monkeypatch.setattr(texturing, "_SPARE_BYTES", 1_000_000)
    monkeypatch.setattr(texturing, "_spare", {})
    yield r
    texturing._spare.clear()


def _call(image_bytes, tex):
    images = [np.zeros((1, image_bytes // 3, 3), np.uint8)]
    return texturing.texture_map_faces(images, (_abi.UguTexFace * 1)(), 1, tex, tex, 3)


def test_kept_while_small(lib):
    for _ in range(3):
        _call(300_000, 100)
    assert lib.created == 1 and not lib.destroyed and len(texturing._spare) == 1


def test_parts_add_up_over_calls(lib):
    _call(700_000, 10)
    assert lib.destroyed == []
    _call(300, 230)  # 13 x 230 x 230 = 687,700 bytes of planes beside the 700,000 of images
    assert lib.destroyed == [1] and not texturing._spare
    _call(300, 230)
    assert lib.created == 2 and lib.destroyed == [1]


def test_not_kept_after_an_error(lib):
    _call(300, 10)
    lib.fail = True
    with pytest.raises(_abi.HipError):
        _call(300, 10)
    assert lib.destroyed == [1] and not texturing._spare


def test_released(lib):
    _call(300, 10)
    texturing._release_spares()
    assert lib.destroyed == [1] and not texturing._spare
