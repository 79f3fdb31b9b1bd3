"""Neighbour-list rows of more tile pairs than one round of a 256-thread block
takes: the persistent kernel, which builds them so, and the step graphs, whose
blocks take 1,024 a round, give the same trajectory bit for bit, with the list
built every step and by the skin rule."""

from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import protein

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("skin", [0.0, 1.5])
def test_rounds_agree(skin):
    from prolix_amd.engine import GBEngine, Langevin

    s = protein(64 * 258 + 1, 77)  # 259 tiles: the first rows take two rounds
    out = []
    for mode in ("graph", "persistent"):
        eng = GBEngine(s, cutoff=12.0, gb_cutoff=True)
        eng.set_nl_skin(skin)
        eng.set_step_mode(mode)
        eng.init(s["positions"], [Langevin(0.5, 300.0, 1.0, seed=4, safety_caps=True)])
        eng.steps(6)
        out.append([a.cpu().numpy() for a in eng.state()])
        eng.close()
    for a, b in zip(*out):
        assert np.isfinite(a).all() and np.array_equal(a, b)
