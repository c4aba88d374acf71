"""The lists and cleared scan results of a load: energies of a rejected
potential read as zero in memory that an earlier batch wrote, at counts around
the cleared chunk, and the other potentials' scans match the oracle."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import oracle
from epseon_backend_amd.workloads import MorseSpec
from tests.helpers import problem_from_spec

pytestmark = pytest.mark.gpu


def _pot(capi, s, levels):
    return capi.Potential(values=s.table(), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.mu, e_top=s.de,
                          n_energies=s.m, level_min=0, level_count=levels)


@pytest.mark.parametrize("m", [1, 63, 65, 4095, 4096, 4097, 12289])
def test_rejected_potentials_read_zero(m):
    from epseon_backend_amd import capi

    sys.stdout.write(f"case: lists of a load, {m} energies\n")
    sys.stdout.flush()
    full = MorseSpec(20.0, 20000.0, 1.7, 1.6, 1.0, 5.0, 500, m)
    small = MorseSpec(20.0, 20000.0, 1.7, 1.6, 1.0, 5.0, 500, 130)
    coarse = MorseSpec(50.0, 40000.0, 2.5, 2.0, 0.2, 9.0, 60, m)
    with capi.Context(0) as ctx:
        t = ctx.tuning()
        t.refine_mode, t.windows = capi.REFINE_SEGMENTED, 1
        ctx.set_tuning(t)
        # Every byte the next load's results may take holds counts and values.
        ctx.load([_pot(capi, full, 3)] * 4)
        ctx.solve(1e-10, 200)
        # The second's grid does not resolve its window: rejected.
        ctx.load([_pot(capi, small, 5), _pot(capi, coarse, 2), _pot(capi, small, 70)])
        assert ctx.potential_info(1).flags != 0
        ctx.solve(1e-10, 200)
        nodes, far, resc = ctx.scan_results()
        levels, status, _ = (a.copy() for a in ctx.levels())
    for a in (nodes, far, resc):
        assert np.all(a[130 : 130 + m] == 0)
    want = oracle.solve(problem_from_spec(small), 0, 5, segmented=True, windows=True)
    for at in (0, 130 + m):
        np.testing.assert_array_equal(nodes[at : at + 130], want[0])
        np.testing.assert_array_equal(far[at : at + 130].view(np.int64), want[1].view(np.int64))
        np.testing.assert_array_equal(resc[at : at + 130], want[2])
    assert np.all(status[:5] == 0) and np.all(status[5:7] == 3)
    np.testing.assert_array_equal(levels[7:12].view(np.int64), levels[:5].view(np.int64))
