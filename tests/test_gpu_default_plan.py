"""The plan of jobs that were not tuned, on both sides of each of its lines, and
their frames against the oracle bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from _helpers import assert_frame_equal, oracle_render, say

pytestmark = pytest.mark.gpu

EYE = np.eye(4, dtype=np.float32).reshape(16)

# width, height, frames -> tile
PLANS = [(80, 24, 1, (16, 16)), (1, 1, 1, (16, 8)), (1020, 240, 1, (16, 16)), (1024, 256, 1, (64, 16)),
         (1024, 256, 13, (64, 16)), (1024, 256, 14, (64, 32)), (81, 25, 1, (16, 8)), (1023, 256, 1, (64, 8)),
         (1023, 256, 13, (64, 8)), (1023, 256, 14, (64, 32)), (65, 40, 300, (64, 8))]


@pytest.mark.parametrize("W,H,frames,tile", PLANS)
def test_tiles(sloth, W, H, frames, tile):
    rng = np.random.default_rng(W + H + frames)
    n = 400
    xy = rng.uniform((0, 0), (max(W / 2, 1), H), (n, 1, 2)) + rng.uniform(-9, 9, (n, 3, 2))
    xyz = np.concatenate([xy, rng.uniform(-1, 1, (n, 3, 1))], 2).astype(np.float32)
    rgb = rng.integers(0, 256, (n, 3), dtype=np.uint8)
    mesh = sloth.SimpleMesh(xyz, rgb)
    b = sloth.Batch([sloth.FrameSpec(W, H, EYE, True) for _ in range(frames)],
                    [sloth.DrawSpec(f, mesh, EYE) for f in range(frames)])
    say(f"case default plan {frames} x {W}x{H}")
    b.run()
    plan = b.plan()
    assert (plan["tile_w"], plan["tile_h"]) == tile
    assert plan["bin_tris_per_thread"] == 1
    ref = oracle_render(W, H, EYE, [(xyz, rgb, EYE, None)])
    for f in {0, frames // 2, frames - 1}:
        cells, z, win = b.read_frame(f, want_winners=True)
        assert_frame_equal(cells, z, win, ref, W)


def test_triangles_per_thread(sloth):
    rng = np.random.default_rng(1)
    n, W, H = 1 << 18, 128, 64
    xy = rng.uniform((0, 0), (W / 2, H), (n, 1, 2)) + rng.uniform(-1, 1, (n, 3, 2))
    xyz = np.concatenate([xy, rng.uniform(-1, 1, (n, 3, 1))], 2).astype(np.float32)
    rgb = rng.integers(0, 256, (n, 3), dtype=np.uint8)
    mesh = sloth.SimpleMesh(xyz, rgb)
    ref = oracle_render(W, H, EYE, [(xyz, rgb, EYE, None)])
    for frames, tpt in ((4, 1), (5, 2), (8, 2), (9, 4)):
        b = sloth.Batch([sloth.FrameSpec(W, H, EYE, True) for _ in range(frames)],
                        [sloth.DrawSpec(f, mesh, EYE) for f in range(frames)])
        say(f"case {frames} x {n} triangles")
        b.run()
        assert b.plan()["bin_tris_per_thread"] == tpt
        cells, z, win = b.read_frame(frames - 1, want_winners=True)
        assert_frame_equal(cells, z, win, ref, W)
        b.set_bin(4)
        b.set_transforms([EYE] * frames)
        assert b.plan()["bin_tris_per_thread"] == 4   # what is set stays
