"""An item's sums are the same on four waves (short work lists) and on two (lists of
5,000 items on): every system of a long list equals itself alone bit for bit, at tile
counts and remainders where halves of columns and rows of patches are empty."""

from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import protein

pytestmark = pytest.mark.gpu

SIZES = (3500, 2300, 1237, 640, 130, 72, 65, 64, 9, 8, 6)  # 2,484 items


@pytest.mark.parametrize("cutoff,gb_cutoff", [(0.0, False), (9.0, False), (12.0, True)])
def test_long_list_equals_each_system_alone(cutoff, gb_cutoff):
    from prolix_amd.engine import GBEngine

    systems = [protein(n, 50 + n % 5) for n in SIZES]

    def run(ss):
        eng = GBEngine(ss, cutoff=cutoff, gb_cutoff=gb_cutoff)
        x = [s["positions"] for s in ss]
        e, f, b = eng.energy_forces(x, born_radii=True)
        out = [a.cpu().numpy() for a in (e, f, b, eng.energy_forces(x, energies=False)[1])]
        eng.close()
        return out

    e, f, b, f0 = run(systems * 3)
    at = 0
    for k, s in enumerate(systems):
        e1, f1, b1, f01 = run([s])
        end = at + len(s["charges"])
        assert np.isfinite(f1).all()
        assert np.array_equal(e[k], e1[0])
        assert np.array_equal(f[at:end], f1) and np.array_equal(f0[at:end], f01) and np.array_equal(b[at:end], b1)
        at = end
