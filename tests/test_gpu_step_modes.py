"""The step kernels at the sizes where they go from four waves per item to two to
one: trajectories equal the captured-graph path's bit for bit, alone and in a pack.

fused: one tile; two; up to 8 items (192 atoms); more. persistent: up to 64 items (640
atoms); up to 150 (1,024 atoms are 136, 1,025 are 153); more."""

from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import protein

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,sizes", [
    ("fused", (8,)), ("fused", (64,)), ("fused", (65,)), ("fused", (128,)), ("fused", (129,)),
    ("fused", (192,)), ("fused", (193,)), ("fused", (321,)),
    ("fused", (40, 64, 9, 64)), ("fused", (64, 128, 65, 9)), ("fused", (64, 65, 192, 193, 520)),
    ("persistent", (640,)), ("persistent", (641,)), ("persistent", (1024,)), ("persistent", (1025,)),
    ("persistent", (300, 641, 64)),
])
def test_equals_graph(mode, sizes):
    from prolix_amd.engine import GBEngine, Langevin

    systems = [protein(n, 60 + n % 9) for n in sizes]
    out = []
    for m in ("graph", mode):
        eng = GBEngine(systems)
        eng.set_step_mode(m)
        eng.init([s["positions"] for s in systems],
                 [Langevin(0.5, 300.0, 1.0, seed=7 + k, safety_caps=True) for k in range(len(systems))])
        eng.steps(12)
        out.append([a.cpu().numpy() for a in eng.state()])
        eng.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)
