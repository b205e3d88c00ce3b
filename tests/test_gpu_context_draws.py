"""A context whose draws change between frames, in number and size: each frame
is that of its own draws, bit for bit."""
from __future__ import annotations

import pytest

from _helpers import assert_frame_equal, oracle_render, say

pytestmark = pytest.mark.gpu


def test_draws_of_other_sizes(sloth):
    from sloth_amd import meshgen

    W, H = 160, 90
    meshes = [meshgen.uv_sphere(12, 6, seed=1), meshgen.uv_sphere(40, 30, seed=2), meshgen.subdivided_box(3, seed=3),
              meshgen.displaced_icosphere(4, seed=4), meshgen.uv_sphere(6, 4, seed=5)]
    sm = [sloth.SimpleMesh.from_mesh(m) for m in meshes]
    U = meshgen.screen_transform(W, H, [m.bbox_max() for m in meshes])
    ctx = sloth.Context(W, H)
    ctx.utransform = U
    for frame, pick in enumerate([(0, 1), (2, 3, 4), (1,), (3, 0), (4, 4, 4, 1, 0, 2), (1, 0), (0, 1)]):
        draws = []
        ctx.clear()
        for k, i in enumerate(pick):
            R = meshgen.rotation_euler(0.2 * k, 0.7 * frame + k, 0.1).copy()
            R[12:14] = 0.3 * (k - 1)
            sloth.draw_mesh(ctx, sm[i], R)
            draws.append((meshes[i].xyz, meshes[i].rgb, R, None))
        say(f"case frame {frame}: draws of meshes {pick}")
        cells, z, win = ctx.read(want_winners=True)
        assert_frame_equal(cells, z, win, oracle_render(W, H, U, draws), W)
