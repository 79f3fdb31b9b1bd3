"""Steps recorded into a caller's own graph (systems up to 192 atoms: the passes
themselves, the fused kernel for one tile and in long calls) and replayed equal
the same steps run directly, bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import protein

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,steps", [(64, 5), (65, 5), (192, 5), (100, 50), (100, 51)])
def test_recorded_steps_equal_direct_ones(n, steps):
    import torch

    from prolix_amd.engine import GBEngine, Langevin

    s = protein(n, 40 + n)
    out = []
    for record in (False, True):
        eng = GBEngine(s)
        eng.init(s["positions"], [Langevin(0.5, 300.0, 1.0, seed=9)])
        torch.cuda.synchronize()
        if record:
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                eng.steps(steps)
        for _ in range(3):
            if record:
                g.replay()
            else:
                eng.steps(steps)
            torch.cuda.synchronize()
            out.append([a.cpu().numpy() for a in eng.state()])
        eng.close()
    for a, b in zip(out[:3], out[3:]):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
