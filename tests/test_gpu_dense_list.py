"""The dense neighbour list at the edges of its tilings (rows per wave, 64-atom
tiles, 64 tiles a scan), complete and with a capacity that overflows."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 257, 4095, 4097])
def test_rows_match_brute_force(n):
    import torch

    from prolix_amd import _native as N

    rng = np.random.default_rng(n)
    x = rng.uniform(0.0, 5.0 + n ** (1.0 / 3.0) * 2.2, (n, 3)).astype(np.float32)
    radius = 6.0
    x64 = x.astype(np.float64)
    d2 = sum((x64[:, None, k] - x64[None, :, k]) ** 2 for k in range(3))
    hit = d2 < radius**2
    near = np.abs(d2 - radius**2) < 36.0 * 4e-7  # float32 may decide these either way
    np.fill_diagonal(hit, False)
    np.fill_diagonal(near, False)
    xd = torch.tensor(x, device="cuda")
    work = torch.empty((8 * ((n + 63) // 64),), dtype=torch.float32, device="cuda")
    full = None
    for cap in (n + 7, 7):
        idx = torch.full((n, cap), -5, dtype=torch.int32, device="cuda")
        counts = torch.full((n,), -5, dtype=torch.int32, device="cuda")
        N.check(N.lib().prx_neighbor_list_dense(*(ctypes.c_void_p(t.data_ptr()) if hasattr(t, "data_ptr") else t
                                                  for t in (xd, n, radius, cap, idx, counts, work)),
                                                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "list")
        got, c = idx.cpu().numpy(), counts.cpu().numpy()
        if full is None:
            full = got
            for i in range(n):
                row = got[i, : c[i]]
                assert np.all(got[i, c[i]:] == n) and np.all(np.diff(row) > 0)
                is_in = np.zeros(n, bool)
                is_in[row] = True
                assert np.array_equal(is_in | near[i], hit[i] | near[i])
            first = c
        else:
            assert np.array_equal(got, full[:, :cap]) and np.array_equal(c, first)
