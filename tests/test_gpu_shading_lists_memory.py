"""When the backward pass's fragment lists take device memory: not before the
first backward pass after a visibility, and not anew for every visibility
that shows a little more."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from _helpers import say

pytestmark = pytest.mark.gpu


def _free_bytes(sloth) -> int:
    sloth.load_library()
    hip = C.CDLL("libamdhip64.so.7")   # the runtime that the library uses
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _scaled(M, s):
    return np.ascontiguousarray((np.asarray(M, np.float32).reshape(4, 4) * np.array([[s], [s], [s], [1]], np.float32)).reshape(16))


def test_lists_are_made_by_the_backward_pass(sloth):
    from sloth_amd import meshgen

    m = meshgen.displaced_icosphere(6, seed=4)
    W = H = 1024
    V = 32
    U = meshgen.screen_transform(W, H, [m.bbox_max()])
    Rs = [meshgen.rotation_euler(0.1, 0.4 * v, 0.2) for v in range(V)]
    mesh = sloth.SimpleMesh.from_mesh(m)
    batch = sloth.Batch([sloth.FrameSpec(W, H, U, True) for _ in range(V)],
                        [sloth.DrawSpec(v, mesh, R) for v, R in enumerate(Rs)])
    n_verts = m.verts.shape[0]
    sh = sloth.Shading(batch, m.faces, n_verts)
    rng = np.random.default_rng(4)
    vc = rng.uniform(0, 1, (n_verts, 3)).astype(np.float32)
    vn = (m.verts / np.linalg.norm(m.verts, axis=1, keepdims=True)).astype(np.float32)
    L = np.array([0.3, -0.5, 0.8], np.float32)
    sh.set_target(np.zeros((V * W * H, 3), np.float32))

    def refresh(s):
        batch.set_transforms(np.stack([_scaled(R, s) for R in Rs]))
        sh.visibility()

    # the largest view first, so that the tile lists have all they will need
    refresh(1.0)
    refresh(0.8)
    sh.forward(vc, vn, L)
    seen = 0
    for v in range(V):
        win = batch.read_frame(v, want_winners=True)[2]
        seen += len(np.unique(win[win >= 0]))
    assert seen > V * 10000
    say("case lists of 32 views")
    before = _free_bytes(sloth)
    sh.backward()
    made = before - _free_bytes(sloth)
    # 16 bytes for each 8 x 8 block of pixels that a triangle shows in: at least
    # one for each triangle seen; the runtime counts in pages of 2 MiB
    assert made > 0 and made >= 16 * seen - (2 << 20)
    for s in (0.82, 0.84, 0.86, 0.88):   # up to a fifth more pixels
        refresh(s)
        held = _free_bytes(sloth)
        sh.backward()
        assert _free_bytes(sloth) == held, s
