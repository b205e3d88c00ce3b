"""Exports of frames of very unlike sizes: the bytes, and the device memory that
the encoder takes, which goes by the stream's cells and not by the number of
frames times the largest."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from _helpers import say

pytestmark = pytest.mark.gpu


def _free_bytes(sloth) -> int:
    sloth.load_library()
    hip = C.CDLL("libamdhip64.so.7")   # the runtime that the library uses
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _export(frames):
    """main.rs:55-58, 85-106 around the frames' flushes."""
    out = b"let frames = [\n"
    for i, t in enumerate(frames):
        out += b"`\n" + t + (b"`,\n" if i + 1 < len(frames) else b"`];\n")
    return out


@pytest.mark.parametrize("order", ["large first", "large last", "alternating", "one large within"])
def test_unlike_frames(sloth, order):
    from sloth_amd import meshgen

    m = meshgen.uv_sphere(10, 5, seed=5)
    mesh = sloth.SimpleMesh.from_mesh(m)
    small, large = [(9 + i % 7, 3 + i % 5) for i in range(40)], [(700, 400), (701, 399), (1200, 800)]
    sizes = {"large first": large + small, "large last": small + large,
             "alternating": [s for i in range(12) for s in (large[i % 3], small[i])],
             "one large within": small[:17] + large[:1] + small[17:]}[order]
    images = [i % 3 != 0 for i in range(len(sizes))]
    Us = [meshgen.screen_transform(W, H, [m.bbox_max()]) for W, H in sizes]
    b = sloth.Batch([sloth.FrameSpec(W, H, U, im) for (W, H), U, im in zip(sizes, Us, images)],
                    [sloth.DrawSpec(f, mesh, meshgen.rotation_euler(0.1 * f, 0.2, 0.0)) for f in range(len(sizes))])
    b.run()
    say(f"case export, {order}")
    for mode in (sloth.ENCODE_HTML, sloth.ENCODE_TEXT):
        texts = [b.encode_frame(f, mode) for f in range(len(sizes))]
        assert b.encode_export(mode=mode) == _export(texts)
        assert b.encode_export(first=3, count=9, mode=mode) == _export(texts[3:12])


def test_memory_of_unlike_frames(sloth):
    W = H = 4096
    n = 3000
    U = np.eye(4, dtype=np.float32).reshape(16)
    b = sloth.Batch([sloth.FrameSpec(8, 8, U, True) for _ in range(n)] + [sloth.FrameSpec(W, H, U, True)], [])
    b.run()
    b.sync()
    say(f"case memory of {n} frames of 8x8 and one of {W}x{H}")
    before = _free_bytes(sloth)
    text = b.encode_export(mode=sloth.ENCODE_TEXT)
    taken = before - _free_bytes(sloth)
    frame = lambda w, h: b"`\n" + b" " * (w * h + h) + b"\n"   # noqa: E731
    assert text == b"let frames = [\n" + (frame(8, 8) + b"`,\n") * n + frame(W, H) + b"`];\n"
    # the stream itself, and 12 bytes a block of 1024 cells (twice over at most),
    # in pages of 2 MiB; 3001 frames of the largest one's blocks are 600 MB
    assert taken <= len(text) + (8 << 20)
