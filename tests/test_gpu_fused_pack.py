"""Many small systems in one engine: the fused kernel steps them side by side,
each at its own pass, and the trajectories equal the captured-graph path's bit
for bit, twice in a row."""

from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import protein

pytestmark = pytest.mark.gpu


def test_fused_pack_equals_graph():
    from prolix_amd.engine import GBEngine, Langevin

    base = [protein(n, 20 + n) for n in (64, 65, 97, 128, 129, 150, 190)]
    systems = [base[k % len(base)] for k in range(98)]
    eng = GBEngine(systems)
    params = [Langevin(0.5, 300.0, 1.0, seed=300 + k, safety_caps=True) for k in range(len(systems))]
    out = []
    for mode in ("graph", "fused", "fused"):
        eng.set_step_mode(mode)
        eng.init([s["positions"] for s in systems], params)
        eng.steps(30)
        out.append([a.cpu().numpy() for a in eng.state()])
    eng.close()
    for got in out[1:]:
        for a, b in zip(out[0], got):
            assert np.array_equal(a, b)
