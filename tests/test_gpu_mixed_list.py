"""Work lists of systems with different shares, short enough for units: units of one,
two and four items (four whole items of a system above 128 tiles, without a
barrier), the last one of a system short of items. Each system's energies and
forces equal bit for bit those of the system alone, whose blocks are others."""

from __future__ import annotations

import numpy as np
import pytest

from tests.helpers import protein

pytestmark = pytest.mark.gpu


# tiles (items): 3 (6), 130 (8,515 = 4 x 2,128 + 3), 41 (861 = 2 x 430 + 1)
@pytest.mark.parametrize("sizes", [(130, 8300, 2600), (8300, 130), (2600, 8300)])
@pytest.mark.parametrize("cutoff,gb_cutoff", [(0.0, False), (9.0, False), (12.0, True)])
def test_systems_of_a_mixed_list_equal_themselves_alone(sizes, cutoff, gb_cutoff):
    from prolix_amd.engine import GBEngine

    systems = [protein(n, 30 + n % 7) for n in sizes]

    def run(ss):
        eng = GBEngine(ss, cutoff=cutoff, gb_cutoff=gb_cutoff)
        x = [s["positions"] for s in ss]
        e, f, _ = eng.energy_forces(x)
        out = e.cpu().numpy(), f.cpu().numpy(), eng.energy_forces(x, energies=False)[1].cpu().numpy()
        eng.close()
        return out

    e, f, f0 = run(systems)
    at = 0
    for k, s in enumerate(systems):
        e1, f1, f01 = run([s])
        end = at + len(s["charges"])
        assert np.array_equal(e[k], e1[0])
        assert np.array_equal(f[at:end], f1) and np.array_equal(f0[at:end], f01)
        at = end
