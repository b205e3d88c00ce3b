"""Read-backs around the sizes at which the copy to the host changes its form
(1 MiB: several threads, 8 MiB: pieces through slots), contexts whose draw
tables grow and shrink between frames, and streams longer than the wrapper's
single-call buffer: everything against the oracle, bit for bit."""
from __future__ import annotations

import threading

import numpy as np
import pytest

import oracle
from _helpers import assert_frame_equal, oracle_render, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(16, 9), (361, 362), (362, 363), (363, 364), (299, 292), (1023, 1024), (1024, 1025),
                                 (1400, 1001)])
def test_read_sizes(sloth, W, H):
    from sloth_amd import meshgen

    m = meshgen.uv_sphere(16, 8, seed=W)
    U = meshgen.screen_transform(W, H, [m.bbox_max()])
    R = meshgen.rotation_euler(0.2, 0.4, 0.1)
    ctx = sloth.Context(W, H)
    ctx.utransform = U
    ctx.clear()
    sloth.draw_mesh(ctx, sloth.SimpleMesh.from_mesh(m), R)
    say(f"case read {W}x{H}")
    ref = oracle_render(W, H, U, [(m.xyz, m.rgb, R, None)])
    cells, z, win = ctx.read()
    assert_frame_equal(cells, z, None, ref, W)
    cells, z, win = ctx.read(want_winners=True)
    assert_frame_equal(cells, z, win, ref, W)
    for mode in (sloth.ENCODE_TEXT, sloth.ENCODE_HTML):
        assert ctx.encode(mode) == oracle.encode(ref.cells, mode)


def test_tables_grow_between_frames(sloth):
    """The tables' pinned copy moves when a frame has more draws than any
    before it; frames before and after are right, read or encoded."""
    from sloth_amd import meshgen

    W, H = 120, 50
    meshes = [meshgen.uv_sphere(12, 6, seed=s) for s in range(3)]
    sm = [sloth.SimpleMesh.from_mesh(m) for m in meshes]
    U = meshgen.screen_transform(W, H, [m.bbox_max() for m in meshes])
    ctx = sloth.Context(W, H)
    ctx.utransform = U
    for n in (1, 2, 9, 1, 40, 3):
        Rs = [meshgen.rotation_euler(0.1 * k, 0.5 + k, 0.2 * n) for k in range(n)]
        say(f"case {n} draws")
        ctx.clear()
        for k, R in enumerate(Rs):
            sloth.draw_mesh(ctx, sm[k % 3], R)
            if k == 0:
                ctx.render()   # a render in flight while the tables grow
        ref = oracle_render(W, H, U, [(meshes[k % 3].xyz, meshes[k % 3].rgb, R, None) for k, R in enumerate(Rs)])
        assert ctx.encode(sloth.ENCODE_ANSI) == oracle.encode(ref.cells, 1)
        cells, z, win = ctx.read(want_winners=True)
        assert_frame_equal(cells, z, win, ref, W)


def test_handles_share_the_pinned_pool(sloth):
    """Contexts on several threads, each made, read and dropped many times:
    every frame is its own."""
    from sloth_amd import meshgen

    m = meshgen.uv_sphere(16, 8, seed=3)
    sm = sloth.SimpleMesh.from_mesh(m)
    sizes = [(64, 20), (400, 300), (700, 500), (90, 33)]
    U = [meshgen.screen_transform(W, H, [m.bbox_max()]) for W, H in sizes]
    R = [meshgen.rotation_euler(0.1, 0.9 * k, 0.3) for k in range(len(sizes))]
    refs = [oracle_render(W, H, U[k], [(m.xyz, m.rgb, R[k], None)]) for k, (W, H) in enumerate(sizes)]
    say("case pool shared by threads")
    bad = []

    def work(k):
        W, H = sizes[k]
        for _ in range(12):
            ctx = sloth.Context(W, H)
            ctx.utransform = U[k]
            ctx.clear()
            sloth.draw_mesh(ctx, sm, R[k])
            cells, z, _ = ctx.read()
            text = ctx.encode(sloth.ENCODE_TEXT)
            if not (np.array_equal(cells, refs[k].cells) and np.array_equal(z.view(np.uint32), refs[k].z.view(np.uint32))
                    and text == oracle.encode(refs[k].cells, 0)):
                bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
