"""An atom at infinity: its pairs' energies are zero, so the pair terms are those of
the same system with the atom very far away (its forces are not numbers, and a bond to
it is infinite). Systems whose last tile is ragged, full, and of one atom.

The pairs at 1e12 A add under 1e-9 kcal/mol and the others are the same float32
numbers in the same FP64 sums: 1e-9 relative to the largest term."""

from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import protein

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [138, 192, 129])
@pytest.mark.parametrize("cutoff", [0.0, 9.0])
def test_pair_energies_are_finite(n, cutoff):
    from prolix_amd import _native as N
    from prolix_amd.engine import GBEngine

    s = protein(n, 70 + n)
    eng = GBEngine([s], cutoff=cutoff)
    out = []
    for far in (1e12, np.inf):
        x = s["positions"].copy()
        x[70] = far
        out.append(eng.energy_forces([x])[0].cpu().numpy()[0])
    eng.close()
    at = [N.TERMS.index(k) for k in ("lj", "gb", "coulomb", "ace")]
    want, got = (e[at] for e in out)
    assert np.isfinite(got).all()
    assert np.abs(got - want).max() <= 1e-9 * np.abs(want).max()
