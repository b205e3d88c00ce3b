"""The work that users of this library have it do, as cases that can be timed and compared.

A case goes through the public entry points of sloth_amd only.  Frames come back as the library keeps
them: cells are 32-bit words and depths are returned as their bit patterns, because the library's contract
for both is bit-exactness; only the shading entry points return computed floats.
"""
from __future__ import annotations

import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(1, os.path.abspath("rust-sloth_amd"))

import sloth_amd  # noqa: E402
from sloth_amd import meshgen  # noqa: E402


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # one frame of the terminal loop: the default terminal, a small model, the colour stream
        {"name": "terminal_80x24", "kind": "terminal", "width": 80, "height": 24, "mesh": "uv", "size": 16},
        # one picture of a model file of four meshes (indexed, as model uploads are), read back to the host
        {"name": "picture_640x480", "kind": "picture", "width": 640, "height": 480, "mesh": "ico", "size": 3,
         "meshes": 4, "indexed": True},
        # the `-j 100` export of a model at 100x100, from render to the finished script
        {"name": "export_100x100", "kind": "export", "width": 100, "height": 100, "frames": 100, "mesh": "ico",
         "size": 3, "indexed": True},
        # an export of a few frames at full picture size
        {"name": "export_1280x720", "kind": "export", "width": 1280, "height": 720, "frames": 4, "mesh": "ico",
         "size": 5, "indexed": False},
        # a thumbnail turntable: many small frames in one replay
        {"name": "sweep_320x240", "kind": "sweep", "width": 320, "height": 240, "frames": 32, "mesh": "ico",
         "size": 4, "indexed": False},
        # the 1080p turntable of the benchmark
        {"name": "sweep_1920x1080", "kind": "sweep", "width": 1920, "height": 1080, "frames": 256, "mesh": "ico",
         "size": 7, "indexed": False},
        # a turntable at an odd width (terminals and windows have any width), from an indexed mesh
        {"name": "sweep_1919x1079", "kind": "sweep", "width": 1919, "height": 1079, "frames": 64, "mesh": "ico",
         "size": 6, "indexed": True},
        # an interactive view of a large mesh: a new transform, one 4K frame
        {"name": "view_3840x2160", "kind": "view", "width": 3840, "height": 2160, "mesh": "ico", "size": 8},
        # a batch of unlike jobs: 30 meshes of 1k to 1M triangles at 80x24 to 2560x1440
        {"name": "jobs_30", "kind": "jobs", "jobs": 30, "least": 1000, "most": 1000000},
        # a serving loop that renders into its own tensors on torch's stream and may not allocate
        {"name": "serve_1280x720", "kind": "serve", "width": 1280, "height": 720, "mesh": "ico", "size": 6},
        # fitting a small model: forward with its picture, then backward
        {"name": "shade_4x512", "kind": "shade", "views": 4, "side": 512, "lon": 64, "lat": 63, "step": False},
        # fitting at full size: one training step over 32 views
        {"name": "shade_32x1024", "kind": "shade", "views": 32, "side": 1024, "lon": 224, "lat": 224, "step": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["terminal", "picture", "export", "sweep", "sweep", "view", "jobs", "serve", "shade", "shade"])
    if kind == "terminal":
        return {"kind": kind, "width": rng.randint(40, 240), "height": rng.randint(12, 70), "mesh": "uv",
                "size": rng.randint(6, 48)}
    if kind == "jobs":
        return {"kind": kind, "jobs": rng.randint(6, 30), "least": 1000, "most": _log(rng, 20000, 1000000)}
    if kind == "shade":
        lon = _log(rng, 24, 224)
        return {"kind": kind, "views": _log(rng, 1, 24), "side": _log(rng, 129, 1024), "lon": lon,
                "lat": max(12, lon + rng.randint(-8, 0)), "step": rng.random() < 0.6}
    height = _log(rng, 100, 2160 if kind == "view" else 1080)
    c = {"kind": kind, "width": int(height * rng.uniform(1.0, 16.0 / 9.0)), "height": height,
         "mesh": rng.choice(["ico", "ico", "box"])}
    slots = c["width"] * c["height"]
    if kind == "picture":
        c.update(meshes=rng.randint(1, 6), indexed=rng.random() < 0.5)
    if kind in ("export", "sweep"):
        most = 4 * 1280 * 720 if kind == "export" else 64 * 1920 * 1080
        c.update(frames=_log(rng, 2, max(2, min(128, most // slots))), indexed=rng.random() < 0.5)
    level = rng.randint(2, 7 if kind in ("sweep", "view") else 6)
    c["size"] = level if c["mesh"] == "ico" else max(1, int(math.sqrt(20 * 4 ** level / 12) * rng.uniform(0.7, 1.4)))
    return c


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _sphere(level):
    return meshgen.icosphere_indexed(level)


@functools.lru_cache(maxsize=None)
def _box(n):
    m = meshgen.subdivided_box(n, 0)
    return m.verts.astype(np.float64), m.faces


@functools.lru_cache(maxsize=None)
def _uv(lon, lat):
    m = meshgen.uv_sphere(lon, lat)
    return m.verts.astype(np.float64), m.faces


def _model(mesh, size, seed, stream=False):
    """(vertices float32, faces, a colour per face) of a seeded model.  Where a character stream comes out
    (stream), the seed draws the colours only, all of three digits, so that every seed's stream is as long."""
    v, f = _sphere(size) if mesh == "ico" else _box(size) if mesh == "box" else _uv(2 * size, size)
    if mesh == "ico":   # bumps, so that triangle sizes vary
        v = v * (1.0 + 0.05 * meshgen.value_noise(v, 1 if stream else seed))[:, None]
    colors = np.random.default_rng(seed).integers(100 if stream else 0, 256, (v.shape[0], 3), dtype=np.uint8)
    return v.astype(np.float32), f, colors[f[:, 0]]


def _upload(model, indexed):
    v, f, c = model
    return sloth_amd.SimpleMesh.indexed(v, f, c) if indexed else sloth_amd.SimpleMesh(v[f], c)


def _triangles(case):
    s = case["size"]
    return 20 * 4 ** s if case["mesh"] == "ico" else 12 * s * s if case["mesh"] == "box" else 4 * s * (s - 1)


def _screen(width, height, model):
    return meshgen.screen_transform(width, height, [np.maximum(model[0].max(axis=0), 0.0)])


def _turntable(frames, rng):
    """A full turn about y from a seeded start, slightly tilted."""
    start, tilt = rng.uniform(0, 2 * math.pi), rng.uniform(-0.3, 0.3)
    return [meshgen.rotation_euler(tilt, float(p), 0.0) for p in meshgen.turntable_pitches(frames, start)]


class _Buffer:
    """A batch's device memory, for torch to view; keeps the batch alive."""

    def __init__(self, owner, address, count):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<i4", "data": (address, False), "version": 3}


def _frames_of(batch):
    """The batch's cells and depths on the device: one tensor each where the frames are alike (their rows then
    lie one pitch apart), else one per frame."""
    def view(address, count):
        return torch.as_tensor(_Buffer(batch, address, count), device="cuda")

    at = [batch.device_frame(i) for i in range(len(batch.frames))]
    n = [(f.width * f.height + (f.height if f.image else 0), f.width * f.height) for f in batch.frames]
    out = []
    for k in (0, 1):
        step = (at[1][k] - at[0][k]) // 4 if len(at) > 1 else n[0][k]
        alike = all(m == n[0] for m in n) and all(a[k] == at[0][k] + 4 * step * i for i, a in enumerate(at))
        if alike:
            whole = view(at[0][k], step * (len(at) - 1) + n[0][k])
            out.append(whole.as_strided((len(at), n[0][k]), (step, 1)))
        else:
            out.append([view(a[k], m[k]) for a, m in zip(at, n)])
    return out


def _jobs(case):
    """Unlike jobs: (mesh kind, size, width, height), in no order of size."""
    rng = np.random.default_rng(case["jobs"])
    got = []
    for i in range(case["jobs"]):
        # counts log-uniform, each stretch of the range met
        share = (i + rng.uniform()) / case["jobs"]
        target = case["least"] * (case["most"] / case["least"]) ** share
        width, height = meshgen.RESOLUTIONS[int(rng.integers(0, len(meshgen.RESOLUTIONS)))]
        if rng.integers(0, 2):
            got.append(("ico", min(range(9), key=lambda k: abs(20 * 4 ** k - target)), width, height))
        else:
            got.append(("box", max(1, round(math.sqrt(target / 12))), width, height))
    return [got[i] for i in rng.permutation(len(got))]


def _shading(case, seed):
    """Everything a fit has in hand: the model, the views, the parameters and a picture to match."""
    v, f = _uv(case["lon"], case["lat"])
    v = v.astype(np.float32)
    rng = np.random.default_rng(seed)
    side, views = case["side"], case["views"]
    gpu = torch.Generator("cuda").manual_seed(seed)
    # the picture: a smooth image with sensor noise, a colour per z slot
    y, x = torch.meshgrid(torch.linspace(0, 6, side, device="cuda"), torch.linspace(0, 6, side, device="cuda"), indexing="ij")
    phase = torch.rand((views, 1, 1, 3), generator=gpu, device="cuda") * 6
    target = 0.5 + 0.4 * torch.sin(x[None, :, :, None] + phase) * torch.cos(y[None, :, :, None] - phase)
    target += 0.02 * torch.randn(target.shape, generator=gpu, device="cuda")
    light = rng.normal(size=3)
    return {"verts": v, "faces": f, "side": side, "views": views,
            "rotations": [meshgen.rotation_euler(*rng.uniform(0, 2 * math.pi, 3)) for _ in range(views)],
            "screen": meshgen.screen_transform(side, side, [np.maximum(v.max(axis=0), 0.0)]),
            "vcolor": rng.uniform(0, 1, v.shape).astype(np.float32),
            "vnormal": (v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32),
            "light": (light / np.linalg.norm(light)).astype(np.float32), "target": target.reshape(-1, 3).float()}


def prepare(case, seed):
    kind, rng = case["kind"], np.random.default_rng(seed)
    if kind == "shade":
        p = _shading(case, seed)
        colors = rng.integers(0, 256, (p["faces"].shape[0], 3), dtype=np.uint8)
        mesh = sloth_amd.SimpleMesh(p["verts"][p["faces"]], colors)
        batch = sloth_amd.Batch([sloth_amd.FrameSpec(p["side"], p["side"], p["screen"]) for _ in p["rotations"]],
                                [sloth_amd.DrawSpec(i, mesh, r) for i, r in enumerate(p["rotations"])])
        fit = sloth_amd.Shading(batch, p["faces"], p["verts"].shape[0])
        fit.set_target(p["target"].cpu().numpy())
        return {"kind": kind, "fit": fit, "step": case["step"], "vcolor": p["vcolor"], "vnormal": p["vnormal"],
                "light": p["light"]}
    if kind == "jobs":
        frames, draws = [], []
        for i, (mesh, size, width, height) in enumerate(_jobs(case)):
            model = _model(mesh, size, seed + i)
            frames.append(sloth_amd.FrameSpec(width, height, _screen(width, height, model)))
            draws.append(sloth_amd.DrawSpec(i, _upload(model, False),
                                            meshgen.rotation_euler(*rng.uniform(0, 2 * math.pi, 3))))
        batch = sloth_amd.Batch(frames, draws)
        return {"kind": kind, "batch": batch, "frames": _frames_of(batch)}

    width, height = case["width"], case["height"]
    stream = kind in ("terminal", "export")
    if stream:
        rng = np.random.default_rng(1)   # the same views for every seed (see _model)
    models = [_model(case["mesh"], case["size"], seed + i, stream) for i in range(case.get("meshes", 1))]
    if kind in ("terminal", "picture"):
        # several meshes: side by side, as the parts of a scene
        for i, (v, f, c) in enumerate(models):
            if len(models) > 1:
                a = 2 * math.pi * i / len(models)
                models[i] = ((v * np.float32(0.5) + np.float32([0.5 * math.cos(a), 0.5 * math.sin(a), 0])), f, c)
        context = sloth_amd.Context(width, height, image=kind == "picture")
        return {"kind": kind, "context": context, "meshes": [_upload(m, case.get("indexed", True)) for m in models],
                "transform": _turntable(1, rng)[0]}
    if kind == "serve":
        v, f, c = models[0]
        return {"kind": kind, "positions": torch.from_numpy(v[f]).cuda(), "colors": torch.from_numpy(c).cuda(),
                "width": width, "height": height, "screen": _screen(width, height, models[0]),
                "transform": _turntable(1, rng)[0],
                "cells": torch.empty(width * height + height, dtype=torch.int32, device="cuda"),
                "depths": torch.empty(width * height, dtype=torch.float32, device="cuda")}
    mesh, screen = _upload(models[0], case.get("indexed", False)), _screen(width, height, models[0])
    turns = _turntable(case.get("frames", 1), rng)
    batch = sloth_amd.Batch([sloth_amd.FrameSpec(width, height, screen) for _ in turns],
                            [sloth_amd.DrawSpec(i, mesh, t) for i, t in enumerate(turns)])
    if kind in ("sweep", "view"):   # plans that are run many times are tuned once
        batch.autotune()
    return {"kind": kind, "batch": batch, "frames": _frames_of(batch), "transforms": np.stack(turns)}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "terminal":
        context = s["context"]
        context.update(s["meshes"])
        context.clear()
        sloth_amd.draw_mesh(context, s["meshes"][0], s["transform"])
        return np.frombuffer(context.encode(sloth_amd.ENCODE_ANSI), np.uint8)
    if kind == "picture":
        context = s["context"]
        context.update(s["meshes"])
        context.clear()
        for mesh in s["meshes"]:
            sloth_amd.draw_mesh(context, mesh, s["transform"])
        cells, depths, _ = context.read()
        return cells.view(np.int32), depths.view(np.int32)
    if kind == "export":
        s["batch"].run()
        return np.frombuffer(s["batch"].encode_export(), np.uint8)
    if kind in ("sweep", "jobs"):
        s["batch"].run()
        return s["frames"]
    if kind == "view":
        s["batch"].set_transforms(s["transforms"])
        s["batch"].run()
        s["batch"].sync()   # the frame is on the screen before the next one is drawn
        return s["frames"]
    if kind == "serve":
        sloth_amd.render_frame_noalloc(s["positions"].data_ptr(), s["colors"].data_ptr(), s["colors"].shape[0], s["width"],
                                       s["height"], True, s["screen"], s["transform"], s["cells"].data_ptr(),
                                       s["depths"].data_ptr(), stream=torch.cuda.current_stream().cuda_stream)
        return s["cells"], s["depths"].view(torch.int32)
    fit = s["fit"]
    if s["step"]:
        loss, d_color, d_normal, d_light = fit.step(s["vcolor"], s["vnormal"], s["light"])
        return {"loss": loss, "d_color": d_color, "d_normal": d_normal, "d_light": d_light}
    loss, picture = fit.forward(s["vcolor"], s["vnormal"], s["light"], want_out=True)
    d_color, d_normal, d_light = fit.backward()
    return {"loss": loss, "picture": picture, "d_color": d_color, "d_normal": d_normal, "d_light": d_light}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _mesh_bytes(case, indexed):
    n = _triangles(case)
    return 15 * n + 12 * (n // 2 + 2) if indexed else 39 * n


def work(case):
    kind = case["kind"]
    if kind == "shade":
        slots, verts = case["views"] * case["side"] ** 2, case["lon"] * (case["lat"] - 1) + 2
        # per slot its winner and target (and its colour out), per triangle its vertex ids, per vertex colour and
        # normal in and their gradients out; about a fifth of the slots is covered
        return {"bytes": slots * (16 if case["step"] else 28) + 24 * verts + 48 * verts, "flops": slots * 0.2 * 150}
    if kind == "jobs":
        got = {"bytes": 0, "flops": 0}
        for mesh, size, width, height in _jobs(case):
            one = work({"kind": "sweep", "mesh": mesh, "size": size, "width": width, "height": height, "frames": 1,
                        "indexed": False})
            got = {k: got[k] + one[k] for k in got}
        return got
    slots = case["width"] * case["height"]
    frames, meshes = case.get("frames", 1), case.get("meshes", 1)
    mesh = meshes * _mesh_bytes(case, case.get("indexed", kind == "terminal"))
    # per triangle the transform, edges and class; per covered pixel (about a fifth) edges, depth and shade
    flops = frames * (meshes * _triangles(case) * 120 + slots * 0.2 * 30)
    if kind in ("terminal", "export"):   # the stream, about 38 bytes a cell
        return {"bytes": mesh + frames * slots * 38, "flops": flops}
    return {"bytes": mesh + frames * (8 * slots + 4 * case["height"]), "flops": flops}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _visible(xyz, faces, side):
    """The winner of each z slot of a side x side picture, in binary32 with each operation rounded by itself (the
    test decides which pixels exist, so it is part of the problem): (slots, triangles, x, y)."""
    t = xyz[faces]
    x, y, z = (t[:, :, k] for k in range(3))
    minx, maxx, miny, maxy = x.amin(1), x.amax(1), y.amin(1), y.amax(1)
    last = float(side - 1)
    x0 = torch.maximum(torch.ceil(minx.clamp(min=1)), torch.floor(minx)).long()
    x1 = torch.minimum(torch.ceil((2 * maxx).clamp(max=last)) - 1, torch.ceil(maxx)).long()
    y0, y1 = torch.ceil(miny.clamp(min=1)).long(), torch.ceil(maxy.clamp(max=last)).long() - 1
    wide, tall = (x1 - x0 + 1).clamp(min=0), (y1 - y0 + 1).clamp(min=0)
    A0, B0 = x[:, 2] - x[:, 1], y[:, 2] - y[:, 1]
    A1, B1 = x[:, 0] - x[:, 2], y[:, 0] - y[:, 2]
    A2, B2 = x[:, 1] - x[:, 0], y[:, 1] - y[:, 0]
    p, q = A2 * (y[:, 2] - y[:, 0]), B2 * (x[:, 2] - x[:, 0])
    a = 1.0 / (p - q)
    count = wide * tall
    tri = torch.repeat_interleave(torch.arange(len(count), device=xyz.device), count)
    at = torch.arange(len(tri), device=xyz.device) - (torch.cumsum(count, 0) - count)[tri]
    ix, iy = x0[tri] + at % wide[tri], y0[tri] + at // wide[tri]
    px, py = ix.float(), iy.float()

    def edge(A, B, k):
        p, q = A[tri] * (py - y[tri, k]), B[tri] * (px - x[tri, k])
        return p - q

    w0, w1, w2 = edge(A0, B0, 1), edge(A1, B1, 2), edge(A2, B2, 0)
    p, q = w1 * (z[:, 1] - z[:, 0])[tri], w2 * (z[:, 2] - z[:, 0])[tri]
    p = a[tri] * (p + q)
    depth = z[tri, 0] + p + 0.0
    hit = (w0 >= 0) & (w1 >= 0) & (w2 >= 0) & (depth < torch.finfo(torch.float32).max)
    tri, ix, iy, depth = tri[hit], ix[hit], iy[hit], depth[hit].contiguous()
    slot = iy * side + 2 * ix
    bits = depth.view(torch.int32).long()
    bits = torch.where(bits < 0, bits ^ 0x7FFFFFFF, bits)   # ordered as the depths are
    key = (bits << 32) | (tri << 1) | (2 * ix < side).long()
    best = torch.full((side * side,), 2 ** 63 - 1, dtype=torch.int64, device=xyz.device)
    best.scatter_reduce_(0, slot, key, "amin")
    won = torch.nonzero(best[slot] == key)[:, 0]
    return slot[won], tri[won], ix[won], iy[won]


def exact(case, seed):
    if case["kind"] != "shade":
        return None   # whole numbers and bytes
    p = _shading(case, seed)
    side, f64 = p["side"], torch.float64
    verts, faces = torch.from_numpy(p["verts"]).cuda(), torch.from_numpy(p["faces"].astype(np.int64)).cuda()
    color, normal, light = (torch.from_numpy(p[k]).cuda().to(f64) for k in ("vcolor", "vnormal", "light"))
    d_color, d_normal, d_light = torch.zeros_like(color), torch.zeros_like(normal), torch.zeros_like(light)
    loss, picture = torch.zeros((), dtype=f64, device="cuda"), []
    target = p["target"].reshape(p["views"], side * side, 3)
    for view in range(p["views"]):
        # utransform * transform and the screen vertices, column by column in binary32
        U, R = p["screen"].reshape(4, 4), p["rotations"][view].reshape(4, 4)   # rows are columns here
        M = np.zeros((4, 4), np.float32)
        for j in range(4):
            M[j] = U[0] * R[j, 0]
            for k in range(1, 4):
                M[j] = U[k] * R[j, k] + M[j]
        m = torch.from_numpy(M).cuda()
        xyz = verts[:, 0:1] * m[0, :3]
        xyz = verts[:, 1:2] * m[1, :3] + xyz
        xyz = verts[:, 2:3] * m[2, :3] + xyz
        xyz = m[3, :3] + xyz
        slot, tri, ix, iy = _visible(xyz, faces, side)
        # from here on in 64 bits
        M64 = torch.from_numpy(U.astype(np.float64).T @ R.astype(np.float64).T).cuda()   # plain rows and columns
        at = (verts.to(f64) @ M64[:3, :3].T + M64[:3, 3])[faces[tri]]
        px, py = ix.to(f64), iy.to(f64)

        def orient(i, j, qx, qy):
            return ((at[:, j, 0] - at[:, i, 0]) * (qy - at[:, i, 1])
                    - (at[:, j, 1] - at[:, i, 1]) * (qx - at[:, i, 0]))

        whole = orient(0, 1, at[:, 2, 0], at[:, 2, 1])
        lam = torch.stack([orient(1, 2, px, py), orient(2, 0, px, py), orient(0, 1, px, py)], 1) / whole[:, None]
        m3 = M64[:3, :3]
        det = torch.linalg.det(m3)
        G = det * torch.linalg.inv(m3).T / det.abs() ** (2.0 / 3.0)
        fv = faces[tri]
        n = (lam[:, :, None] * (normal[fv] @ G.T)).sum(1)
        c = (lam[:, :, None] * color[fv]).sum(1)
        shade = n @ light
        out = shade[:, None] * c
        r = out - target[view][slot].to(f64)
        loss += (r * r).sum()
        g = 2 * r
        d_shade = (g * c).sum(1)
        for k in range(3):
            d_color.index_add_(0, fv[:, k], lam[:, k:k + 1] * shade[:, None] * g)
            d_normal.index_add_(0, fv[:, k], (d_shade * lam[:, k])[:, None] * (G.T @ light))
        d_light += d_shade @ n
        if not case["step"]:
            whole_picture = torch.zeros((side * side, 3), dtype=f64, device="cuda")
            whole_picture[slot] = out
            picture.append(whole_picture)
    got = {"loss": float(loss), "d_color": d_color, "d_normal": d_normal, "d_light": d_light}
    if not case["step"]:
        got["picture"] = torch.cat(picture)
    return got
