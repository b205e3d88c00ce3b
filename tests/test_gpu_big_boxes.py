"""Boxes of many tiles and many pixels, in the direct and the wrapped region and
across both, against the oracle bit for bit, winners included; and blocks of
small triangles whose tiles form every shape of the binning window, within it
and past it."""
from __future__ import annotations

import numpy as np
import pytest

from _helpers import assert_frame_equal, oracle_render, say

pytestmark = pytest.mark.gpu

EYE = np.eye(4, dtype=np.float32).reshape(16)


def _check(b, f, W, H, xyz, rgb):
    cells, z, win = b.read_frame(f, want_winners=True)
    assert_frame_equal(cells, z, win, oracle_render(W, H, EYE, [(xyz, rgb, EYE, None)]), W)


@pytest.mark.parametrize("walk", [0, 1])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 300])
@pytest.mark.parametrize("W,tile", [(320, (64, 32)), (320, (16, 8)), (322, (256, 16)), (319, (64, 16)), (321, (32, 8))])
def test_big_triangles(sloth, W, tile, n, walk):
    H = 150
    rng = np.random.default_rng(n + W)
    c = rng.uniform((0, 0), (W, H), (n, 2))   # past W / 2: the wrapped region
    xy = c[:, None, :] + rng.uniform(-1, 1, (n, 3, 2)) * rng.uniform(5, 110, (n, 1, 1))
    xyz = np.concatenate([xy, rng.uniform(-1, 1, (n, 3, 1))], 2).astype(np.float32)
    rgb = rng.integers(0, 256, (n, 3), dtype=np.uint8)
    b = sloth.Batch([sloth.FrameSpec(W, H, EYE, True)], [sloth.DrawSpec(0, sloth.SimpleMesh(xyz, rgb), EYE)])
    b.set_tile(*tile)
    b.set_walk(walk)
    say(f"case big triangles {W}x{H}, {n} triangles, tile {tile}, walk {walk}")
    for _ in range(2):
        b.run()
        _check(b, 0, W, H, xyz, rgb)


SHAPES = [(1, 60), (60, 1), (16, 16), (17, 30), (32, 16), (33, 15), (33, 8), (33, 17), (64, 8), (65, 4), (64, 64)]


@pytest.mark.parametrize("tpt", [1, 2, 4])
@pytest.mark.parametrize("side", ["direct", "wrapped", "across"])
def test_windows(sloth, side, tpt):
    """A block's small triangles spread over w x h tiles of 8 x 4 cells."""
    W, H, n = 600, 262, 1300
    frames, draws, parts = [], [], []
    for i, (w, h) in enumerate(SHAPES):
        rng = np.random.default_rng(i)
        left = {"direct": 4, "wrapped": W / 2 + 4, "across": W / 2 - 2 * w}[side]
        c = rng.uniform((left, 3), (left + 4 * w - 4, 4 * h - 1), (n, 2))
        xy = c[:, None, :] + rng.uniform(-2, 2, (n, 3, 2))
        xyz = np.concatenate([xy, rng.uniform(-1, 1, (n, 3, 1))], 2).astype(np.float32)
        rgb = rng.integers(0, 256, (n, 3), dtype=np.uint8)
        frames.append(sloth.FrameSpec(W, H, EYE, True))
        draws.append(sloth.DrawSpec(i, sloth.SimpleMesh(xyz, rgb), EYE))
        parts.append((xyz, rgb))
    b = sloth.Batch(frames, draws)
    b.set_tile(8, 4)
    b.set_bin(tpt)
    say(f"case binning windows: {side}, {tpt} triangles a thread")
    b.run()
    for f, (xyz, rgb) in enumerate(parts):
        _check(b, f, W, H, xyz, rgb)


@pytest.mark.parametrize("tall", [10, 255, 256, 700])
def test_tall_among_many(sloth, tall):
    """Draws of different sizes, one of them of tall triangles."""
    rng = np.random.default_rng(tall)
    frames, draws, parts = [], [], []
    for f, (W, H, n, s) in enumerate([(320, 200, 70000, 1.5), (160, 700, tall, 60.0), (128, 90, 3000, 4.0)]):
        xy = rng.uniform((0, 0), (W / 2, H), (n, 1, 2)) + rng.uniform(-s, s, (n, 3, 2))
        xyz = np.concatenate([xy, rng.uniform(-1, 1, (n, 3, 1))], 2).astype(np.float32)
        rgb = rng.integers(0, 256, (n, 3), dtype=np.uint8)
        frames.append(sloth.FrameSpec(W, H, EYE, True))
        draws.append(sloth.DrawSpec(f, sloth.SimpleMesh(xyz, rgb), EYE))
        parts.append((W, H, xyz, rgb))
    b = sloth.Batch(frames, draws)
    say(f"case {tall} tall triangles among many")
    b.run()
    for f, p in enumerate(parts):
        _check(b, f, *p)
