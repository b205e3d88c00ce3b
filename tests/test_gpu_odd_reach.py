"""Odd widths whose wrapped boxes reach further from run to run, and back: the
columns of the raster's odd instance grow with room to spare, and every frame
equals the oracle's."""
from __future__ import annotations

import numpy as np
import pytest

from _helpers import assert_frame_equal, oracle_render, say

pytestmark = pytest.mark.gpu


def _moved(R, tx):
    M = np.asarray(R, np.float32).reshape(4, 4).copy()
    M[3, 0] = tx   # column-major: the translation's x
    return np.ascontiguousarray(M.reshape(16))


@pytest.mark.parametrize("tile", [None, (16, 8), (128, 16)])
def test_reach_grows(sloth, tile):
    from sloth_amd import meshgen

    m = meshgen.displaced_icosphere(3, seed=6)
    small = meshgen.uv_sphere(10, 5, seed=1)
    W, H = 361, 92
    U = meshgen.screen_transform(W, H, [m.bbox_max()])
    R0, R1 = meshgen.rotation_euler(0.3, 0.2, 0.0), meshgen.rotation_euler(0.0, 1.1, 0.4)
    meshes = [sloth.SimpleMesh.from_mesh(m), sloth.SimpleMesh.from_mesh(small)]
    frames = [sloth.FrameSpec(W, H, U, True), sloth.FrameSpec(W, H, U, False), sloth.FrameSpec(W + 1, H, U, True)]
    b = sloth.Batch(frames, [sloth.DrawSpec(f, meshes[k], R) for f in range(3) for k, R in ((0, R0), (1, R1))])
    if tile:
        b.set_tile(*tile)
    for tx in (0.0, 0.3, 0.7, 1.1, 1.6, 2.4, 0.2, 3.0, -0.5, 2.0):
        Rs = [_moved(R0, tx), _moved(R1, tx * 0.5)]
        say(f"case reach, tile {tile}, x {tx}")
        b.set_transforms(np.stack(Rs * 3))
        b.run()
        b.sync()
        for f, fs in enumerate(frames):
            ref = oracle_render(fs.width, H, U, [(m.xyz, m.rgb, Rs[0], None), (small.xyz, small.rgb, Rs[1], None)],
                                image=fs.image)
            cells, z, win = b.read_frame(f, want_winners=True)
            assert_frame_equal(cells, z, win, ref, fs.width)
