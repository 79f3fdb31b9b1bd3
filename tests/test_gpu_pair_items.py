"""The pair passes at the edges of their tilings: patches of 8, tiles of 64, the
sizes at which items go from four shares to two to whole, and the work list's
length at which a wave takes an item instead of a group of waves a unit.

Tolerances as everywhere: energy 1e-6 and force RMS 1e-5 relative to the
float64 oracle on the same float32 inputs. The two ways to run an item give
the same sums bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import gb_oracle as O
from tests.helpers import protein, rel_rms

pytestmark = pytest.mark.gpu


def _evaluate(systems, **kw):
    from prolix_amd.engine import GBEngine

    eng = GBEngine(systems, **kw)
    e, f, _ = eng.energy_forces([s["positions"] for s in systems], energies=True)
    f0 = eng.energy_forces([s["positions"] for s in systems], energies=False)[1]
    out = e.cpu().numpy(), f.cpu().numpy(), f0.cpu().numpy()
    eng.close()
    return out


@pytest.mark.parametrize("n", [64, 65, 71, 72, 73, 127, 128, 2560, 2561])
@pytest.mark.parametrize("cutoff", [0.0, 9.0])
def test_edges_match_the_oracle(n, cutoff):
    s = protein(n, 900 + n)
    e, f, f0 = _evaluate([s], cutoff=cutoff)
    terms = O.energy_terms(s, s["positions"], cutoff=cutoff)
    scale = max(abs(terms["total"]), 0.2 * sum(abs(terms[k]) for k in O.TERM_NAMES))
    assert abs(e[0][-1] - terms["total"]) <= 1e-6 * scale
    fo = O.forces(s, s["positions"], cutoff=cutoff)
    assert rel_rms(f, fo) <= 1e-5 and rel_rms(f0, fo) <= 1e-5


@pytest.mark.parametrize("cutoff,gb_cutoff", [(0.0, False), (12.0, True)])
def test_waves_and_units_agree(cutoff, gb_cutoff):
    """Systems of four, two and one share per item, alone (units) and in a pack of
    more than 64,000 items (a wave each)."""
    systems = [protein(n, 30 + n % 7) for n in (130, 2300, 2600, 8300, 130)]
    systems += [systems[3]] * 7
    e, f, f0 = _evaluate(systems, cutoff=cutoff, gb_cutoff=gb_cutoff)
    at = 0
    for k, s in enumerate(systems[:5]):
        n = len(s["charges"])
        e1, f1, f01 = _evaluate([s], cutoff=cutoff, gb_cutoff=gb_cutoff)
        assert np.array_equal(e[k], e1[0]), n
        assert np.array_equal(f[at:at + n], f1), n
        assert np.array_equal(f0[at:at + n], f01), n
        at += n
