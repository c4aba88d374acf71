"""Refinement in 128- and 256-lane blocks through their segment tables: levels
and iteration counts bit-identical to the natural table (a load under the
64-lane setting builds none for wider blocks) and to the oracle, on grids whose
segments have even, odd and uneven step counts and at the table's threshold."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import oracle
from epseon_backend_amd.workloads import MorseSpec
from tests.helpers import problem_from_spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("windows", [0, 1])
@pytest.mark.parametrize("lanes", [128, 256])
def test_wide_tables_match_natural_table_and_oracle(lanes, windows):
    from epseon_backend_amd import capi

    sys.stdout.write(f"case: {lanes} lanes, windows {windows}\n")
    sys.stdout.flush()
    # 64 to 67 steps per lane, all equal and uneven; then short grids with
    # fewer segments than lanes.
    sizes = [64 * lanes + 2, 64 * lanes + 3, 65 * lanes + 1, 65 * lanes + 2, 67 * lanes + 2, 16_384, 16_385,
             32 * lanes - 5, 700]
    specs = [MorseSpec(20.0 + i, 20000.0, 1.7, 1.6, 1.0, 5.0, n, 300) for i, n in enumerate(sizes)]
    pots = [capi.Potential(values=s.table(), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.mu, e_top=s.de,
                           n_energies=s.m, level_min=0, level_count=12) for s in specs]
    got = []
    for load_lanes in (lanes, 64):
        with capi.Context(0) as ctx:
            t = ctx.tuning()
            t.refine_mode, t.windows, t.segmented_lanes = capi.REFINE_SEGMENTED, windows, load_lanes
            ctx.set_tuning(t)
            ctx.load(pots)
            t.segmented_lanes = lanes
            ctx.set_tuning(t)
            ctx.solve(1e-10, 200)
            assert ctx.stats().refine_lanes == lanes
            got.append(tuple(a.copy() for a in ctx.levels()))
    for a, b in zip(*got):
        np.testing.assert_array_equal(a.view(np.int32), b.view(np.int32))
    levels, status, iterations = got[0]
    assert np.all(status == 0)
    for i in (2, 4, 8):
        want = oracle.solve(problem_from_spec(specs[i]), 0, 12, 1e-10, 200, segmented=True, lanes=lanes,
                            windows=bool(windows))
        np.testing.assert_array_equal(levels[12 * i:12 * i + 12].view(np.int64), want[3].view(np.int64))
        np.testing.assert_array_equal(iterations[12 * i:12 * i + 12], want[4])
