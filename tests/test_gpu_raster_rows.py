"""The tile raster's rows and stores where they can go wrong, against the
oracle bit for bit: lists of one chunk (256 entries), one more and several, in
which winners' cells are put aside between chunks; shaders whose glyph must be
evaluated per pixel; zero depths of either sign; depths that are huge,
infinite or NaN; boxes from one to many columns; widths of every residue
modulo 4."""
from __future__ import annotations

import numpy as np
import pytest

from _helpers import assert_frame_equal, oracle_render, say

pytestmark = pytest.mark.gpu

SHADERS = {"default": None,
           "unsorted": dict(thresholds=(0.6, 0.2, 0.9, 0.4), glyphs="abcd", fallback="z")}


def _soup(n, W, H, seed, size, depths):
    """n triangles over the frame, edges up to `size` pixels, either facing,
    depths drawn from `depths`."""
    rng = np.random.default_rng(seed)
    c = rng.uniform((1, 1), (W / 2 - 1, H - 1), (n, 2))
    p = c[:, None, :] + rng.uniform(-size, size, (n, 3, 2))
    z = rng.choice(np.asarray(depths, np.float32), (n, 3))
    xyz = np.concatenate([p, z[..., None]], 2).astype(np.float32)
    return xyz, rng.integers(0, 256, (n, 3), dtype=np.uint8)


def _matrices():
    """Identities whose depth row's other entries are -0, so that a depth of
    -0 stays -0."""
    m = np.eye(4, dtype=np.float32)
    m[2, :] = [-0.0, -0.0, 1.0, -0.0]
    return m.T.reshape(16).copy(), m.T.reshape(16).copy()   # column-major


def _check(sloth, W, H, xyz, rgb, shader, tile, walk):
    U, R = _matrices()
    sh = sloth.Shader(**shader) if shader else sloth.default_shader
    mesh = sloth.SimpleMesh(xyz, rgb)
    b = sloth.Batch([sloth.FrameSpec(W, H, U, True)], [sloth.DrawSpec(0, mesh, R)], sh)
    b.set_tile(*tile)
    b.set_walk(walk)
    b.run()
    cells, z, win = b.read_frame(0, want_winners=True)
    ref = oracle_render(W, H, U, [(xyz, rgb, R, shader and sh)], image=True)
    assert_frame_equal(cells, z, win, ref, W)
    return z


@pytest.mark.parametrize("walk", [0, 1])
@pytest.mark.parametrize("shader", list(SHADERS))
@pytest.mark.parametrize("n", [255, 256, 257, 512, 513, 1400])
def test_chunks(sloth, n, shader, walk):
    W, H = 64, 32   # one tile
    xyz, rgb = _soup(n, W, H, seed=n, size=6, depths=np.linspace(-1, 1, 37))
    say(f"case rows: {n} entries, {shader} shader, walk {walk}")
    _check(sloth, W, H, xyz, rgb, SHADERS[shader], (64, 32), walk)


@pytest.mark.parametrize("walk", [0, 1])
@pytest.mark.parametrize("shader", list(SHADERS))
@pytest.mark.parametrize("n", [40, 256, 900])
def test_zero_depths(sloth, n, shader, walk):
    """Depths that are or round to +0 and -0 (a first vertex at -0 and the
    others a denormal below it): which of two zeros is stored is the
    first-drawn triangle's, with its sign."""
    W, H = 62, 40
    xyz, rgb = _soup(n, W, H, seed=3 * n, size=9, depths=[0.0, -0.0, -0.0, 1e-30])
    xyz[::3, 0, 2] = -0.0
    xyz[::3, 1:, 2] = -1.4e-45
    xyz[1::3, :, 2] = 0.0
    say(f"case zero depths: {n} entries, {shader} shader, walk {walk}")
    z = _check(sloth, W, H, xyz, rgb, SHADERS[shader], (64, 32), walk)
    bits = z.view(np.uint32)
    assert (bits == 0x80000000).any() and (bits == 0).any()


@pytest.mark.parametrize("walk", [0, 1])
@pytest.mark.parametrize("n", [60, 700])
def test_extreme_depths(sloth, n, walk):
    W, H = 64, 48
    big = np.float32(3.4e38)
    xyz, rgb = _soup(n, W, H, seed=n + 1, size=8,
                     depths=[0.5, -0.5, 1e20, -1e20, big, -big, np.inf, -np.inf, np.nan, 2.0 ** 60, 2.0 ** 59])
    xyz[::2, :, 2] = np.float32(0.25)   # half of them plain, so that wavefronts mix
    say(f"case extreme depths: {n} entries, walk {walk}")
    _check(sloth, W, H, xyz, rgb, None, (64, 32), walk)


@pytest.mark.parametrize("W", [60, 61, 62, 63, 64, 65, 66, 130, 131])
@pytest.mark.parametrize("size", [0.7, 2.5, 5.0, 30.0])
def test_widths_and_box_columns(sloth, W, size):
    """Boxes of 1 to 60 columns; frames whose rows start at every residue of
    16 bytes; partial tiles and last slot pairs."""
    H = 50
    xyz, rgb = _soup(500, W, H, seed=int(W + 10 * size), size=size, depths=np.linspace(-3, 3, 61))
    say(f"case columns: width {W}, edges to {size}")
    for tile in ((16, 8), (64, 32)):
        for walk in (0, 1):
            _check(sloth, W, H, xyz, rgb, None, tile, walk)
