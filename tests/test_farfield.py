"""The far-field polynomials as the pair kernels run them: float32 coefficients
scaled so that the leading one is exactly 1 (Born) or -4 (chain), with s^3/3 of the
atom in front. Their error against the series is what the header states, and for
every tier no more than the float32 polynomials of the widest one."""

from __future__ import annotations

import re
from pathlib import Path

import numpy as np
import pytest

HEADER = Path(__file__).resolve().parent.parent / "prolix_amd/csrc/prx_obc_farfield.h"
TIERS = {"": 0, "4": 1, "3": 2, "2": 3}  # suffix -> place of its error line


def _series(y, chain):
    return sum(2 * k * ((k + 1) if chain else 1) / (2 * k + 1) * y ** (k - 1) for k in range(1, 300))


@pytest.mark.parametrize("suffix", TIERS)
@pytest.mark.parametrize("name,scale,lead", [("H", 1.5, 1.0), ("K", -3.0, -4.0)])
def test_error_of_the_polynomial_that_runs(suffix, name, scale, lead):
    txt = HEADER.read_text()
    c = [float(v.rstrip("f")) for v in re.search(rf"kObc{name}{suffix}\[\d+\] = \{{(.*?)\}}", txt).group(1).split(",")]
    xmax = float(re.search(rf"PRX_OBC_FAR{suffix}_XMAX ([0-9.]+)f", txt).group(1))
    stated = re.findall(r"max relative error: h ([0-9.e-]+), k ([0-9.e-]+)", txt)[TIERS[suffix]][name == "K"]
    used = np.float32(scale * np.array(c)).astype(np.float64)
    assert used[0] == lead
    y = np.linspace(0.0, xmax**2, 40001)
    err = np.max(np.abs(np.polyval(used[::-1], y) / (scale * _series(y, name == "K")) - 1.0))
    assert err <= 1.01 * float(stated)
    assert err <= (3.2e-8 if name == "H" else 1.5e-8)
