"""Two atoms at the same point, in different tiles: what the pair gives is not a
number, and stays with the two. Every other atom's force is the oracle's, and
with safety caps (a non-finite force counts as zero) it is not zeroed either.

Tolerance as everywhere: force RMS 1e-5 relative to the float64 oracle."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import gb_oracle as O
from prolix_amd import synth
from tests.helpers import protein, rel_rms

pytestmark = pytest.mark.gpu

TILE = 64


def _coincident(n, ti, tj):
    """A protein with an atom of tile tj moved onto one of tile ti, a pair in which
    neither descreens the other (so that its Born integrals are zero)."""
    s = protein(n, n, radius=synth.compact_radius(n))
    rho, sr = s["radii"] - O.DIELECTRIC_OFFSET, s["scaled_radii"]
    for i in range(TILE * ti, TILE * (ti + 1)):
        for j in range(min(n, TILE * (tj + 1)) - 1, TILE * tj - 1, -1):
            if sr[i] < rho[j] and sr[j] < rho[i] and j > i + 30:
                s["positions"] = s["positions"].copy()
                s["positions"][j] = s["positions"][i]
                return s, np.isin(np.arange(n), (i, j), invert=True)
    raise AssertionError("no such pair")


# four shares an item, the last tile ragged and full; two shares
@pytest.mark.parametrize("n,ti,tj", [(190, 0, 2), (1024, 3, 11), (2600, 1, 39)])
def test_other_atoms_keep_their_forces(n, ti, tj):
    from prolix_amd.engine import GBEngine, Langevin

    s, others = _coincident(n, ti, tj)
    want = O.forces(s, s["positions"])[others]
    eng = GBEngine([s])
    for energies in (True, False):
        f = eng.energy_forces([s["positions"]], energies=energies)[1].cpu().numpy()[others]
        assert np.isfinite(f).all()
        assert rel_rms(f, want) <= 1e-5
    eng.init(s["positions"], [Langevin(1.0, 300.0, 1.0, seed=1, safety_caps=True)])
    f = eng.state()[2].cpu().numpy()[others]
    eng.close()
    free = np.linalg.norm(want, axis=1) < 9000.0  # below the force cap of 10,000
    assert free.sum() > n // 2
    assert np.sqrt(np.mean((f - want)[free] ** 2)) <= 1e-5 * np.sqrt(np.mean(want**2))
