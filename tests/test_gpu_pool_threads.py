"""Contexts made, read, encoded and dropped on several threads at once, which
share the pinned pool: every call succeeds and every frame is its own.  An
error in any thread fails the test (Future.result raises it)."""
from __future__ import annotations

from concurrent.futures import ThreadPoolExecutor

import pytest

import oracle
from _helpers import assert_frame_equal, oracle_render, say

pytestmark = pytest.mark.gpu

SIZES = [(64, 20), (400, 300), (700, 500), (90, 33), (1400, 1001)]
ROUNDS = 8


def test_threads_share_the_pinned_pool(sloth):
    from sloth_amd import meshgen

    m = meshgen.uv_sphere(16, 8, seed=3)
    sm = sloth.SimpleMesh.from_mesh(m)
    U = [meshgen.screen_transform(W, H, [m.bbox_max()]) for W, H in SIZES]
    R = [meshgen.rotation_euler(0.1, 0.9 * k, 0.3) for k in range(len(SIZES))]
    refs = [oracle_render(W, H, U[k], [(m.xyz, m.rgb, R[k], None)]) for k, (W, H) in enumerate(SIZES)]
    texts = [oracle.encode(r.cells, 0) for r in refs]

    def work(k):
        W, H = SIZES[k]
        for n in range(ROUNDS):
            ctx = sloth.Context(W, H)
            ctx.utransform = U[k]
            ctx.clear()
            sloth.draw_mesh(ctx, sm, R[k])
            cells, z, win = ctx.read(want_winners=n % 2 == 1)
            assert_frame_equal(cells, z, win, refs[k], W, check_win=n % 2 == 1)
            assert ctx.encode(sloth.ENCODE_TEXT) == texts[k]
        return ROUNDS

    say(f"case {len(SIZES)} threads")
    with ThreadPoolExecutor(len(SIZES)) as ex:
        done = [f.result(timeout=100) for f in [ex.submit(work, k) for k in range(len(SIZES))]]
    assert done == [ROUNDS] * len(SIZES)
