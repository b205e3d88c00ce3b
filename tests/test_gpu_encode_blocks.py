"""The stream encoder at the edges of its blocks (1024 cells), of the small
single-launch form (16,384 cells) and of its device groups (256 MiB), byte
for byte against the oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from _helpers import say

pytestmark = pytest.mark.gpu


def _batch(sloth, sizes, shader=None):
    """One frame per (W, H, image), a coarse mesh in each."""
    from sloth_amd import meshgen

    m = meshgen.uv_sphere(16, 8, seed=11)   # colours of one to three digits
    sm = sloth.SimpleMesh.from_mesh(m)
    frames = [sloth.FrameSpec(W, H, meshgen.screen_transform(W, H, [m.bbox_max()]), image) for W, H, image in sizes]
    draws = [sloth.DrawSpec(f, sm, meshgen.rotation_euler(0.1 * f, 0.7 + f, 0.3)) for f in range(len(sizes))]
    b = sloth.Batch(frames, draws, shader) if shader else sloth.Batch(frames, draws)
    b.run()
    b.sync()
    return b


@pytest.mark.parametrize("W,H,image", [(1, 1, False), (1, 1, True), (3, 1, False), (33, 31, False), (32, 32, False),
                                       (41, 25, False), (40, 25, True), (64, 64, True), (241, 17, False),
                                       (128, 128, False), (145, 113, False), (128, 127, True), (128, 128, True),
                                       (200, 110, True)])
def test_block_edges(sloth, W, H, image):
    sh = sloth.Shader((0.3, 0.6, 1.0), "·x@", "é")   # one- and two-byte chars
    b = _batch(sloth, [(W, H, image)], sh)
    cells, _, _ = b.read_frame(0)
    say(f"case encode blocks {W}x{H} image={image}: {cells.size} cells")
    for mode in (sloth.ENCODE_TEXT, sloth.ENCODE_ANSI, sloth.ENCODE_HTML):
        assert b.encode_frame(0, mode) == oracle.encode(cells, mode, image=image)
    for mode in (sloth.ENCODE_TEXT, sloth.ENCODE_HTML):
        want = b"let frames = [\n`\n" + oracle.encode(cells, mode, image=image) + b"`];\n"
        assert b.encode_export(mode=mode) == want


def test_export_of_unlike_frames(sloth):
    """Frames of different sizes and modes in one export, whole and in part,
    and the buffer's checks."""
    import ctypes as C

    sizes = [(80, 24, False), (200, 150, True), (1, 1, True), (129, 65, True), (1024, 33, False), (31, 33, True)]
    b = _batch(sloth, sizes)
    cells = [b.read_frame(f)[0] for f in range(len(sizes))]
    say("case export of unlike frames")
    for mode in (sloth.ENCODE_TEXT, sloth.ENCODE_HTML):
        for first, count in ((0, len(sizes)), (1, 3), (4, 1), (5, 1), (2, 4)):
            want = b"let frames = [\n"
            for f in range(first, first + count):
                want += b"`\n" + oracle.encode(cells[f], mode, image=sizes[f][2])
                want += b"`,\n" if f + 1 < first + count else b"`];\n"
            assert b.encode_export(first, count, mode) == want
            L, n = sloth.load_library(), C.c_uint64()
            short = C.create_string_buffer(len(want) - 1)
            assert L.sloth_batch_encode_export(b._h, first, count, mode, short, len(want) - 1, C.byref(n)) == 1
            exact = C.create_string_buffer(len(want) + 1)   # the byte after the stream stays as it was
            exact[len(want)] = b"\x5a"
            assert L.sloth_batch_encode_export(b._h, first, count, mode, exact, len(want), C.byref(n)) == 0
            assert n.value == len(want) and exact.raw == want + b"\x5a"


def test_export_of_several_groups(sloth):
    """An export past 256 MiB leaves the device in groups of whole frames:
    every frame's bytes are those of its own flush."""
    b = _batch(sloth, [(1920, 1080, True)] * 4)
    say("case export of several groups")
    got = b.encode_export()
    assert len(got) > (256 << 20)
    at = len(b"let frames = [\n")
    assert got[:at] == b"let frames = [\n"
    for f in range(4):
        one = b.encode_frame(f, sloth.ENCODE_HTML)
        framed = b"`\n" + one + (b"`,\n" if f < 3 else b"`];\n")
        assert got[at:at + len(framed)] == framed
        at += len(framed)
    assert at == len(got)
    cells, _, _ = b.read_frame(3)
    assert one == oracle.encode(cells, 2)
