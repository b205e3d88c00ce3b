"""The stages of a profiled render on the general path: each kernel's time
under its own name, whichever width parity the batch has."""
from __future__ import annotations

import numpy as np
import pytest

from _helpers import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,runs,idle", [(1280, ["k_finish_global"], ["k_winner_global", "k_resolve_global"]),
                                         (1279, ["k_winner_global", "k_resolve_global"], ["k_finish_global"])])
def test_stage_names(sloth, monkeypatch, W, runs, idle):
    from sloth_amd import meshgen

    monkeypatch.setenv("SLOTH_FORCE_GLOBAL", "1")
    m = meshgen.displaced_icosphere(4, seed=2)
    U = meshgen.screen_transform(W, 720, [m.bbox_max()])
    mesh = sloth.SimpleMesh.from_mesh(m)
    F = 48
    b = sloth.Batch([sloth.FrameSpec(W, 720, U, True) for _ in range(F)],
                    [sloth.DrawSpec(f, mesh, meshgen.rotation_euler(0.0, 0.1 * f, 0.0)) for f in range(F)])
    say(f"case stages of {F} frames of {W}x720")
    b.run()
    b.sync()
    times = [b.profile() for _ in range(5)]
    assert set(times[0]) == {"k_clear_global", "k_raster_global", "k_finish_global", "k_winner_global", "k_resolve_global"}
    least = {k: np.min([t[k] for t in times]) for k in times[0]}
    # 44 million cells: a kernel that runs takes tens of microseconds, two
    # events with nothing between them a few
    assert min(least[k] for k in runs) > 2 * max(least[k] for k in idle)
