"""The raster's bound on the terms of its constant-glyph proof: over the box of
a triangle (box_x of sloth_device.h: within a pixel of the vertices' x extent,
inside their y extent) the edge terms and the orient's own sum to at most
wy (6 wx + 2), wx and wy the extents."""
import numpy as np


def test_terms_bound():
    rng = np.random.default_rng(4)
    n = 200000
    scale = np.exp(rng.uniform(np.log(0.05), np.log(300), (n, 1, 1)))
    aspect = np.exp(rng.uniform(-4, 4, (n, 1)))
    v = rng.uniform(0, 1000, (n, 1, 2)) + rng.normal(size=(n, 3, 2)) * scale
    v[:, :, 1] = v[:, :1, 1] + (v[:, :, 1] - v[:, :1, 1]) * aspect
    v = v.astype(np.float32)
    x, y = v[..., 0], v[..., 1]
    f32 = np.float32
    wx, wy = x.max(1) - x.min(1), y.max(1) - y.min(1)
    bound = wy * (f32(6) * wx + f32(2))
    # the widest box of the two classes, and every row of the extent
    X0, X1 = np.floor(x.min(1)), np.ceil(x.max(1))
    Y0, Y1 = np.ceil(y.min(1)), np.ceil(y.max(1)) - 1
    has = Y0 <= Y1
    terms = np.zeros(n)
    for a, b, k in ((1, 2, 1), (2, 0, 2), (0, 1, 0)):   # edge a -> b anchored at vertex k
        A, B = (x[:, b] - x[:, a]).astype(np.float64), (y[:, b] - y[:, a]).astype(np.float64)
        dy = np.maximum(abs(Y0 - y[:, k].astype(np.float64)), abs(Y1 - y[:, k].astype(np.float64)))
        dx = np.maximum(abs(X0 - x[:, k].astype(np.float64)), abs(X1 - x[:, k].astype(np.float64)))
        terms += abs(A) * dy + abs(B) * dx
    x64, y64 = x.astype(np.float64), y.astype(np.float64)
    terms += abs(x64[:, 1] - x64[:, 0]) * abs(y64[:, 2] - y64[:, 0]) + abs(y64[:, 1] - y64[:, 0]) * abs(x64[:, 2] - x64[:, 0])
    assert has.sum() > n // 2
    # roundings of the bound itself (a few 2^-24) are within the proof's margin
    assert (terms[has] <= bound[has].astype(np.float64) * (1 + 1e-6)).all()
