"""Refinements in 128- and 256-lane blocks with more than two wavefronts per
SIMD give the bits of those with fewer, through the segment tables and the
natural table, and the oracle's."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import oracle
from epseon_backend_amd.workloads import MorseSpec
from tests.helpers import problem_from_spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("longest", [4_000, 16_384])
@pytest.mark.parametrize("lanes", [128, 256])
def test_large_batches_equal_small_ones(lanes, longest):
    from epseon_backend_amd import capi

    sys.stdout.write(f"case: {lanes} lanes, up to {longest} points\n")
    sys.stdout.flush()
    specs = [MorseSpec(20.0 + 0.1 * i, 20000.0, 1.7, 1.6, 1.0, 5.0, longest if i == 0 else 700 + 5 * i, 128)
             for i in range(260)]
    pots = [capi.Potential(values=s.table(), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.mu, e_top=s.de,
                           n_energies=s.m, level_min=0, level_count=9) for s in specs]
    got = []
    # 2,340 levels are 4,680 or 9,360 wavefronts; 45 are 90 or 180.
    for part in (260, 5):
        with capi.Context(0) as ctx:
            t = ctx.tuning()
            t.refine_mode, t.windows, t.segmented_lanes = capi.REFINE_SEGMENTED, 1, lanes
            ctx.set_tuning(t)
            ctx.load(pots[:part])
            ctx.solve(1e-10, 200)
            assert ctx.stats().refine_lanes == lanes
            got.append(tuple(a.copy() for a in ctx.levels()))
    for a, b in zip(*got):
        np.testing.assert_array_equal(a[:45].view(np.int32), b.view(np.int32))
    levels, status, iterations = got[0]
    assert np.all(status == 0)
    for i in (0, 7, 259):
        want = oracle.solve(problem_from_spec(specs[i]), 0, 9, 1e-10, 200, segmented=True, lanes=lanes, windows=True)
        np.testing.assert_array_equal(levels[9 * i:9 * i + 9].view(np.int64), want[3].view(np.int64))
        np.testing.assert_array_equal(iterations[9 * i:9 * i + 9], want[4])
