"""The general path's last pass at widths of either parity, against the oracle
bit for bit: frames of one and two columns, wrapped pixels on the newline cell's
row, empty scenes, both modes, and cell buffers that start at any 4-byte
address."""
from __future__ import annotations

import numpy as np
import pytest

from _helpers import assert_frame_equal, oracle_render, say
from test_zz_no_alloc import _Dev

pytestmark = pytest.mark.gpu

EYE = np.eye(4, dtype=np.float32).reshape(16)


@pytest.mark.parametrize("image", [True, False])
@pytest.mark.parametrize("n", [0, 1, 255, 257])
def test_widths(sloth, n, image):
    dev = _Dev(sloth)
    try:
        for W, H in [(1, 5), (2, 1), (2, 7), (3, 4), (4, 1), (6, 300), (31, 9), (32, 9), (254, 3), (258, 5)]:
            rng = np.random.default_rng(W * 1000 + n)
            # centres over the frame's domain and beyond its logical width
            xyz = np.concatenate([rng.uniform((0, 0), (W, H), (n, 2))[:, None, :] + rng.uniform(-4, 4, (n, 3, 2)),
                                  rng.uniform(-1, 1, (n, 3, 1))], 2).astype(np.float32)
            rgb = rng.integers(0, 256, (n, 3), dtype=np.uint8)
            say(f"case general path {W}x{H}, image {image}, {n} triangles")
            nc = W * H + (H if image else 0)
            d_xyz, d_rgb = dev.upload(xyz), dev.upload(rgb)
            d_cells, d_z = dev.upload(np.full(nc + 3, 7, np.uint32)), dev.upload(np.full(W * H + 3, 7, np.uint32))
            sloth.render_frame_noalloc(d_xyz, d_rgb, n, W, H, image, EYE, EYE, d_cells + 4, d_z + 4)
            cells, z = dev.download(d_cells, nc + 3, np.uint32), dev.download(d_z, W * H + 3, np.float32)
            for a, m in ((cells, nc), (z.view(np.uint32), W * H)):   # nothing outside the frame is written
                assert a[0] == 7 and (a[m + 1:] == 7).all()
            ref = oracle_render(W, H, EYE, [(xyz, rgb, EYE, None)] if n else [], image=image)
            assert_frame_equal(cells[1:nc + 1], z[1:W * H + 1], None, ref, W)
            dev.free()
    finally:
        dev.free()
