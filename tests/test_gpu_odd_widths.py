"""Frames of odd width, against the oracle bit for bit, winners included: boxes
that end before, at and past the last cell column (its slots' second cells are
the next rows' first, wrapped pixels land on odd columns), at widths on both
sides of the tiles' edges; and transforms that move a mesh over that column and
back after the lists were sized."""
from __future__ import annotations

import numpy as np
import pytest

from _helpers import assert_frame_equal, oracle_render, say

pytestmark = pytest.mark.gpu

EYE = np.eye(4, dtype=np.float32).reshape(16)


def _soup(n, x0, x1, H, seed, size):
    """n triangles about points of [x0, x1] x [0, H), clipped to x <= x1."""
    rng = np.random.default_rng(seed)
    p = rng.uniform((x0, 0), (max(x0, x1), H), (n, 2))[:, None, :] + rng.uniform(-size, size, (n, 3, 2))
    p[..., 0] = np.minimum(p[..., 0], x1)
    z = rng.uniform(-1, 1, (n, 3, 1))
    return np.concatenate([p, z], 2).astype(np.float32), rng.integers(0, 256, (n, 3), dtype=np.uint8)


def _shift(dx):
    m = np.eye(4, dtype=np.float32)
    m[0, 3] = dx
    return m.T.reshape(16).copy()   # column-major


# the right end of the boxes, in logical pixels from W / 2 (the last column's)
REACH = {"inside": -1.6, "last": 0.4, "wrapped": 3.0, "far": 40.0}


@pytest.mark.parametrize("walk", [0, 1])
@pytest.mark.parametrize("reach", list(REACH))
@pytest.mark.parametrize("W", [1, 3, 5, 7, 15, 17, 31, 33, 63, 65, 67, 127, 129])
def test_reach(sloth, W, reach, walk):
    H, x1 = 21, W // 2 + REACH[reach]
    for tile, n, size, image in (((16, 8), 300, 4, True), ((64, 16), 40, 12, False), ((8, 4), 9, 30, True)):
        xyz, rgb = _soup(n, 0, x1, H, seed=W + n, size=size)
        b = sloth.Batch([sloth.FrameSpec(W, H, EYE, image)], [sloth.DrawSpec(0, sloth.SimpleMesh(xyz, rgb), EYE)])
        b.set_tile(*tile)
        b.set_walk(walk)
        say(f"case odd width {W}, {reach}, tile {tile}, walk {walk}")
        ref = oracle_render(W, H, EYE, [(xyz, rgb, EYE, None)], image=image)
        for _ in range(2):   # each render leaves its tables as the next expects them
            b.run()
            cells, z, win = b.read_frame(0, want_winners=True)
            assert_frame_equal(cells, z, win, ref, W)


def test_degenerate_triangles(sloth):
    """Boxes computed apart (slivers and triangles that cover their whole
    domain) at the last column and past it."""
    W, H = 65, 30
    rng = np.random.default_rng(5)
    a = rng.uniform((0, 0), (40, H), (60, 2))
    xyz = np.zeros((60, 3, 3), np.float32)
    xyz[:, 0, :2] = a
    xyz[:, 1, :2] = a + (rng.uniform(1, 9, (60, 1)) * (1, 1))
    xyz[:, 2, :2] = a + (rng.uniform(1, 9, (60, 1)) * (1, 1))
    xyz[..., 2] = rng.uniform(-1, 1, (60, 3))
    rgb = rng.integers(0, 256, (60, 3), dtype=np.uint8)
    b = sloth.Batch([sloth.FrameSpec(W, H, EYE, True)], [sloth.DrawSpec(0, sloth.SimpleMesh(xyz, rgb), EYE)])
    say("case odd width: degenerate triangles")
    b.run()
    cells, z, win = b.read_frame(0, want_winners=True)
    assert_frame_equal(cells, z, win, oracle_render(W, H, EYE, [(xyz, rgb, EYE, None)]), W)


@pytest.mark.parametrize("sizes", [[(65, 20)], [(65, 20), (33, 20), (64, 20)], [(129, 33), (1, 9), (40, 12)]])
def test_moves_over_the_edge(sloth, sizes):
    """Frames of one or several widths; every step's transform is new to the
    sized lists, and the synchronising call renders again where needed."""
    frames, draws, parts = [], [], []
    for f, (W, H) in enumerate(sizes):
        xyz, rgb = _soup(200, 0, W // 2 - 6, H, seed=f, size=5)
        frames.append(sloth.FrameSpec(W, H, EYE, True))
        draws.append(sloth.DrawSpec(f, sloth.SimpleMesh(xyz, rgb), EYE))
        parts.append((W, H, xyz, rgb))
    b = sloth.Batch(frames, draws)
    for dx in (0, 4.5, 5.5, 7, 12, 30, 0, 6, 5, -3):
        m = _shift(dx)
        b.set_transforms([m] * len(draws))
        say(f"case odd widths {sizes}: moved by {dx}")
        b.run()
        for f, (W, H, xyz, rgb) in enumerate(parts):
            cells, z, win = b.read_frame(f, want_winners=True)
            assert_frame_equal(cells, z, win, oracle_render(W, H, EYE, [(xyz, rgb, m, None)]), W)
