"""Boxes of many tiles and many pixels, in the direct and the wrapped region and
across both, against the oracle bit for bit, winners included."""
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
