"""Counts of a cumulative mass whose descent ends before its last level: bins that hold one entry at each of the levels, entries
one bit apart, an exact hit of the threshold.  Bit-exact against the oracle."""

import numpy as np
import pytest
import torch

from oracle import shareprefill_oracle as O

pytestmark = pytest.mark.gpu


def test_cover_count_of_bins_with_one_entry(gpu_device):
    from shareprefill_amd import ops

    rng = np.random.default_rng(5)
    rows = []
    rows.append(2.0 ** -np.arange(1, 33))                        # an exponent each: the first level decides
    rows.append(0.25 + np.arange(32) * 2.0 ** -9)                # apart by the second level's bits
    rows.append(0.25 + np.arange(32) * 2.0 ** -16)               # ... by the third's
    rows.append(0.25 + np.arange(32) * 2.0 ** -25)               # ... by the last bit
    rows.append(np.repeat(0.25 + np.arange(16) * 2.0 ** -9, 2))  # two entries in every bin
    rows.append(np.repeat([0.5, 0.25, 0.125, 2.0 ** -20], 8))    # ties and powers of two: thresholds that are hit exactly
    rows += [rng.random(32) ** 8 for _ in range(20)]
    x = np.stack(rows).astype(np.float32)
    for n in (1, 2, 3, 31, 32):
        part = np.ascontiguousarray(x[:, :n])
        for thr in (0.25, 0.5, 0.75, 1.0, 3.0, float(np.nextafter(np.float32(0.75), np.float32(0))), 1e-6):
            got = ops.cover_count(torch.from_numpy(part).to(gpu_device), thr).cpu().tolist()
            assert got == [O.cover_count(row, thr) for row in part], (n, thr)
