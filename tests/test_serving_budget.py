"""The serving loop's footprint of a work item covers what the engine allocates for one."""

from __future__ import annotations

from prolix_amd.serving import hbm_bytes

# 2 x 64 float4 partials, item, unit, three FP64 energies, class
ITEM = 2 * 64 * 16 + 32 + 8 + 3 * 8 + 4


def test_item_bytes():
    tiles = (40, 80)
    items = [t * (t + 1) // 2 for t in tiles]
    per_atom = hbm_bytes(64) - hbm_bytes(0) - (hbm_bytes(1) - hbm_bytes(0))  # 63 atoms more in one tile
    lo, hi = (hbm_bytes(64 * t) - 64 * t * per_atom // 63 for t in tiles)
    assert (hi - lo) / (items[1] - items[0]) >= ITEM
