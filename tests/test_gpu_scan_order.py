"""Task order of the windowed scan: bins that end inside, at and before the part
that is ordered longest first give every trial energy the same shot."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from epseon_backend_amd import capi, workloads

pytestmark = pytest.mark.gpu


# 64-lane tasks per XCD: 32 x 9 = 288 of equal grids, 128 x 9 = 1,152 (past the
# ordered part), and ragged grids with a partly filled last wavefront.
@pytest.mark.parametrize("count,points,energies", [(256, 9_001, 513), (1024, 9_001, 576), (300, 0, 1_999)])
def test_windowed_scan_equals_single_potentials(count, points, energies):
    specs = [dataclasses.replace(s, n=points or max(s.n, 8_000), m=energies) for s in workloads.batched(count)]
    pots = [capi.Potential(values=s.table(), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.mu, e_top=s.de,
                           n_energies=s.m, level_min=0, level_count=1) for s in specs]
    ctx = capi.Context(0)
    t = ctx.tuning()
    t.windows = 1
    ctx.set_tuning(t)
    ctx.load(pots)
    ctx.scan()
    assert ctx.stats().scan_windows == 1
    got = [np.array(x).reshape(count, energies) for x in ctx.scan_results()]
    for p in (0, 1, count // 2, count - 2, count - 1):
        ctx.load(pots[p:p + 1])
        ctx.scan()
        for x, y in zip(got, ctx.scan_results()):
            np.testing.assert_array_equal(x[p], np.array(y))
    ctx.close()
