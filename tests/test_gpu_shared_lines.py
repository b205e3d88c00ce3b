"""Tiles whose rows share memory lines with the tiles beside them (widths that
are no multiples of 32 cells, tiles 64 wide) and those that do not, one width
to a batch and several, against the oracle bit for bit, winners included."""
from __future__ import annotations

import numpy as np
import pytest

from _helpers import assert_frame_equal, oracle_render, say

pytestmark = pytest.mark.gpu

EYE = np.eye(4, dtype=np.float32).reshape(16)


def _mesh(sloth, W, H, n, seed):
    rng = np.random.default_rng(seed)
    xy = rng.uniform((0, 0), (W / 2 + 3, H), (n, 1, 2)) + rng.uniform(-4, 4, (n, 3, 2))
    xyz = np.concatenate([xy, rng.uniform(-1, 1, (n, 3, 1))], 2).astype(np.float32)
    rgb = rng.integers(0, 256, (n, 3), dtype=np.uint8)
    return xyz, rgb, sloth.SimpleMesh(xyz, rgb)


@pytest.mark.parametrize("tile", [None, (64, 8), (64, 32), (32, 16), (128, 16)])
@pytest.mark.parametrize("widths", [[w] for w in (62, 64, 66, 94, 96, 98, 126, 128, 130, 190, 194)] +
                         [[63], [65], [161], [64, 66], [128, 62, 191], [96, 160]])
def test_widths(sloth, widths, tile):
    frames, draws, parts, meshes = [], [], [], []
    # frames after one another, at every alignment; without a tile, as many as
    # the default plan takes tiles of 64 x 32 cells for
    for f in range(2 * len(widths) + 1 if tile else 900):
        W, H = widths[f % len(widths)], 41
        if f >= 2 * len(widths) + 1:
            xyz, rgb, mesh = parts[f % (2 * len(widths))][2:4] + (meshes[f % (2 * len(widths))],)
        else:
            xyz, rgb, mesh = _mesh(sloth, W, H, 90 + 400 * (f % 2), f)
        meshes.append(mesh)
        frames.append(sloth.FrameSpec(W, H, EYE, f % 3 != 0))
        draws.append(sloth.DrawSpec(f, mesh, EYE))
        parts.append((W, H, xyz, rgb, f % 3 != 0))
    b = sloth.Batch(frames, draws)
    if tile:
        b.set_tile(*tile)
    say(f"case widths {widths}, tile {tile}")
    assert tile or (b.plan()["tile_w"], b.plan()["tile_h"]) == (64, 32)
    for walk in (0, 1):
        b.set_walk(walk)
        b.run()
        for f, (W, H, xyz, rgb, image) in list(enumerate(parts))[::1 if tile else 131]:
            cells, z, win = b.read_frame(f, want_winners=True)
            assert_frame_equal(cells, z, win, oracle_render(W, H, EYE, [(xyz, rgb, EYE, None)], image=image), W)
