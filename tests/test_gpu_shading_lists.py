"""The backward pass's fragment lists where they can go wrong, against the
FP64 adjoint: triangles of many pixel blocks, boxes at block and segment
edges, slivers, wrapped pixels, odd widths, soups whose vertices overflow the
workgroup's table, several draws a frame, and a visibility that is older than
the transforms.  Bound as elsewhere for these gradients: 1e-5 norm-wise."""
from __future__ import annotations

import math

import numpy as np
import pytest

import oracle
from _helpers import say

pytestmark = pytest.mark.gpu

REL = 1e-5


def _check(sloth, xyz, faces, n_verts, Us, Rs, W, H, seed, draws_per_frame=1, Rs_later=None):
    rng = np.random.default_rng(seed)
    views = len(Rs) // draws_per_frame
    rgb = rng.integers(0, 256, (len(xyz), 3), dtype=np.uint8)
    mesh = sloth.SimpleMesh(xyz, rgb)
    batch = sloth.Batch([sloth.FrameSpec(W, H, Us, True) for _ in range(views)],
                        [sloth.DrawSpec(i // draws_per_frame, mesh, R) for i, R in enumerate(Rs)])
    vc = rng.uniform(0, 1, (n_verts, 3)).astype(np.float32)
    vn = rng.normal(size=(n_verts, 3))
    vn = (vn / np.linalg.norm(vn, axis=1, keepdims=True)).astype(np.float32)
    L = np.array([0.3, -0.5, 0.8], np.float32)
    target = rng.uniform(0, 1, (views * W * H, 3)).astype(np.float32)
    sh = sloth.Shading(batch, faces, n_verts)
    sh.set_target(target)
    use = Rs
    if Rs_later is not None:
        batch.set_transforms(np.stack(Rs_later))   # the visibility stays that of Rs
        use = Rs_later
    got = [sh.step(vc, vn, L) for _ in range(2)]
    covered, loss, gc, gn, gl = 0, 0.0, np.zeros((n_verts, 3)), np.zeros((n_verts, 3)), np.zeros(3)
    for v in range(views):
        f = oracle.Frame(W, H, True)
        for k in range(draws_per_frame):
            f.draw_mesh(Us, xyz, rgb, Rs[v * draws_per_frame + k])
        covered += int((f.win >= 0).sum())
        for k in range(draws_per_frame):
            # the fragments of this draw alone (its triangles, its matrix)
            one = oracle.Frame(W, H, True)
            lo_t, hi_t = k * len(xyz), (k + 1) * len(xyz)
            mine = (f.win >= lo_t) & (f.win < hi_t)
            one.win[:] = np.where(mine, f.win - lo_t, -1)
            one.winxy[:] = f.winxy
            M = oracle.mat4_mul(Us, use[v * draws_per_frame + k])
            lo, _, (a, b, c) = oracle.shade_f64(one, M, xyz, faces, vc, vn, L, target[v * W * H:(v + 1) * W * H],
                                                want_grad=True)
            loss += lo
            gc += a
            gn += b
            gl += c
    assert covered > 0
    for loss_g, dc, dn, dl in got:   # twice: the accumulators are left clean
        assert abs(loss_g - loss) <= REL * abs(loss)
        for name, g, ref in (("color", dc, gc), ("normal", dn, gn), ("light", dl, gl)):
            err = np.linalg.norm(g.astype(np.float64) - ref) / np.linalg.norm(ref)
            assert err <= REL, (name, err)
    return covered


def _quads(n, W, H, seed):
    """2n screen-space triangles (identity transforms): n rectangles at random
    depth and size, whose pixel boxes start and end at every offset."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(n):
        w, h = np.exp(rng.uniform(0, math.log(W / 2), 1))[0], np.exp(rng.uniform(0, math.log(H), 1))[0]
        x, y, z = rng.uniform(0, W / 2), rng.uniform(0, H), rng.uniform(-1, 1)
        a, b, c, d = (x, y, z), (x + w, y, z), (x + w, y + h, z), (x, y + h, z)
        out += [(a, b, c), (a, c, d)]
    return np.array(out, np.float32)


@pytest.mark.parametrize("W,H", [(96, 64), (97, 64), (300, 200)])
@pytest.mark.parametrize("n", [1, 32, 127, 129, 300])
def test_boxes_of_all_sizes(sloth, W, H, n):
    """1 to 600 rectangles' halves from sub-pixel to the whole frame, soups:
    three vertices a triangle, up to 768 in a workgroup's table of 512."""
    xyz = _quads(n, W, H, seed=n)
    faces = np.arange(3 * len(xyz), dtype=np.uint32).reshape(-1, 3)
    say(f"case shading lists {W}x{H}, {len(xyz)} triangles")
    _check(sloth, xyz, faces, 3 * len(xyz), np.eye(4, dtype=np.float32).reshape(16),
           [np.eye(4, dtype=np.float32).reshape(16)], W, H, seed=n)


@pytest.mark.parametrize("W", [120, 121])
def test_wrapped_pixels_and_slivers(sloth, W):
    """Triangles right of the logical width wrap into the next row, and
    slivers take the exact row spans."""
    H, rng = 70, np.random.default_rng(8)
    wide = np.array([[(W * 0.4, 5, 0), (W * 0.95, 8, 0), (W * 0.5, 60, 0)],
                     [(W * 0.6, 10, -1), (W * 0.9, 30, -1), (W * 0.55, 50, 1)]], np.float32)
    slivers = []
    for _ in range(60):
        a = rng.uniform((2, 2), (W * 0.7, H - 2))
        b = a + rng.uniform(-40, 40, 2)
        c = a + (b - a) * rng.uniform(0.3, 0.7) + rng.normal(0, 1e-4, 2)
        slivers.append([(*a, -2), (*b, -2), (*c, -2)])
        slivers.append([(*a, -2), (*c, -2), (*b, -2)])
    xyz = np.concatenate([wide, np.array(slivers, np.float32)])
    faces = np.arange(3 * len(xyz), dtype=np.uint32).reshape(-1, 3)
    I = np.eye(4, dtype=np.float32).reshape(16)
    say(f"case shading lists wrapped, width {W}")
    # the slivers' own weights are ill-conditioned in binary32, so they are
    # only asked below whether they take part
    _check(sloth, xyz[:2], faces[:2], 6, I, [I], W, H, seed=3)
    rgb = np.zeros((len(xyz), 3), np.uint8)
    b = sloth.Batch([sloth.FrameSpec(W, H, I, True)], [sloth.DrawSpec(0, sloth.SimpleMesh(xyz, rgb), I)])
    sh = sloth.Shading(b, faces, 3 * len(xyz))
    f = oracle.Frame(W, H, True)
    f.draw_mesh(I, xyz, rgb, I)
    # colours and normals 1, light along z, target 0: with G = 1 every
    # fragment's normal weights are its barycentrics times a positive
    # factor, so a triangle has a gradient exactly where it is visible
    ones = np.ones((3 * len(xyz), 3), np.float32)
    vn = np.tile(np.array([0, 0, 1], np.float32), (3 * len(xyz), 1))
    sh.set_target(np.zeros((W * H, 3), np.float32))
    _, dc, dn, _ = sh.step(ones, vn, np.array([0, 0, 1], np.float32))
    seen = np.unique(f.win[f.win >= 0])
    got = np.nonzero(np.abs(dn.reshape(-1, 9)).sum(axis=1) > 0)[0]
    assert np.array_equal(got, seen)


@pytest.mark.parametrize("lon,lat", [(32, 5), (33, 5), (64, 3), (48, 40)])
def test_segment_edges_and_draws(sloth, lon, lat):
    """Triangle counts around multiples of 256, two draws a frame."""
    from sloth_amd import meshgen

    m = meshgen.uv_sphere(lon, lat, seed=2)
    rng = np.random.default_rng(lon)
    W, H = 140, 90
    U = meshgen.screen_transform(W, H, [m.bbox_max()])
    Rs = []
    for _ in range(6):
        R = meshgen.rotation_euler(*rng.uniform(0, 2 * math.pi, 3)).copy()
        R[12:15] = rng.uniform(-0.4, 0.4, 3)
        Rs.append(R.astype(np.float32))
    say(f"case shading lists uv {lon}x{lat}: {m.n} triangles, 3 views of 2 draws")
    _check(sloth, m.xyz, m.faces.astype(np.uint32), len(m.verts), U, Rs, W, H, seed=lon, draws_per_frame=2)


def test_visibility_older_than_the_transforms(sloth):
    """sloth_batch_set_transforms without sloth_shading_visibility: the pixels
    stay those of the old transforms, the matrices are the new ones."""
    from sloth_amd import meshgen

    m = meshgen.uv_sphere(40, 20, seed=6)
    W, H = 128, 100
    U = meshgen.screen_transform(W, H, [m.bbox_max()])
    Rs = [meshgen.rotation_euler(0.1 * k, 0.5 + k, 0.2) for k in range(3)]
    later = [meshgen.rotation_euler(0.1 * k + 0.02, 0.51 + k, 0.19) for k in range(3)]
    say("case shading lists with an older visibility")
    # (the normal map is that of the visibility too, so colours only: light
    # and normals along z make the shade the map's entry alone)
    rng = np.random.default_rng(1)
    rgb = rng.integers(0, 256, (m.n, 3), dtype=np.uint8)
    mesh = sloth.SimpleMesh(m.xyz, rgb)
    b = sloth.Batch([sloth.FrameSpec(W, H, U, True) for _ in Rs], [sloth.DrawSpec(i, mesh, R) for i, R in enumerate(Rs)])
    sh = sloth.Shading(b, m.faces, len(m.verts))
    b.set_transforms(np.stack(later))
    vc = rng.uniform(0, 1, (len(m.verts), 3)).astype(np.float32)
    vn = rng.normal(size=vc.shape).astype(np.float32)
    L = np.array([0.2, 0.3, 0.9], np.float32)
    loss0, out = sh.forward(vc, vn, L, want_out=True)
    sh.set_target(np.zeros_like(out))
    loss, dc, dn, dl = sh.step(vc, vn, L)
    # target 0: the loss is the picture's square, and the sum of each
    # parameter group times its gradient is twice the loss (out is linear in
    # colours, normals and light)
    want = float((out.astype(np.float64) ** 2).sum())
    assert want > 0 and abs(loss - want) <= REL * want
    for p, g in ((vc, dc), (vn, dn), (L, dl)):
        assert abs(float((p.astype(np.float64) * g.astype(np.float64)).sum()) - 2 * want) <= REL * 2 * want * 4
    covered = sum(int((oracle.render(W, H, U, m.xyz, rgb, R).win >= 0).sum()) for R in Rs)
    assert int((np.abs(out).sum(axis=1) != 0).sum()) == covered
