"""The bracket pass over grids of 1 to 4,097 energies (around the sizes of its
search rounds and of its rows of lanes) against the oracle's bracket_level from
the same scan arrays, bit for bit, and the statistics summed from the levels."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import oracle
from epseon_backend_amd.workloads import MorseSpec
from tests.helpers import problem_from_spec

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 4, 5, 15, 16, 17, 63, 64, 65, 255, 256, 257, 4097]


@pytest.mark.parametrize("copies", [1, 9])
@pytest.mark.parametrize("windows", [0, 1])
def test_bracket_rows(windows, copies):
    from epseon_backend_amd import capi

    sys.stdout.write(f"case: brackets, windows {windows}, {copies} copies\n")
    sys.stdout.flush()
    # Two levels more than the well holds; the last are in no bracket.
    specs = [MorseSpec(20.0, 20000.0, 1.7, 1.6, 1.0, 5.0, 701, m) for m in SIZES] * copies
    counts = [s.bound_levels() + 2 for s in specs]
    pots = [capi.Potential(values=s.table(), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.mu, e_top=s.de,
                           n_energies=s.m, level_min=0, level_count=c) for s, c in zip(specs, counts)]
    with capi.Context(0) as ctx:
        t = ctx.tuning()
        t.refine_mode, t.windows = capi.REFINE_SEGMENTED, windows
        ctx.set_tuning(t)
        ctx.load(pots)
        ctx.solve(1e-10, 200)
        nodes, far, resc = ctx.scan_results()
        br = ctx.brackets()
        levels, status, iterations = (a.copy() for a in ctx.levels())
        stats = ctx.stats()
    assert stats.levels_converged == int(np.sum(status == 0))
    if not windows:
        assert stats.refine_point_updates == float(np.sum(np.maximum(iterations, 0).astype(np.int64)) * (701 - 2))
    eo = lo = 0
    for i, s in enumerate(specs[: len(SIZES)]):
        prob = problem_from_spec(s)
        win = prob.windows(bool(windows))
        fe = oracle.band_far_exps(win)
        nd, fr, rs = nodes[eo : eo + s.m], far[eo : eo + s.m], resc[eo : eo + s.m]
        for v in range(counts[i]):
            ref = oracle.bracket_level(nd, fr, rs, prob.e_lo, prob.e_top, v, fe, win)
            got = br[lo + v]
            assert int(got["found"]) == ref.found, (s.m, v)
            if ref.found:
                assert np.float64(got["e_hi"]).view(np.int64) == np.float64(ref.e_hi).view(np.int64), (s.m, v)
                assert np.float64(got["e_lo"]).view(np.int64) == np.float64(ref.e_lo).view(np.int64), (s.m, v)
                assert (int(got["nodes_lo"]), int(got["nodes_hi"]), int(got["lo_valid"]), int(got["band"])) == (
                    ref.c_lo, ref.c_hi, ref.lo_valid, ref.band), (s.m, v)
        want = oracle.solve(prob, 0, counts[i], 1e-10, 200, segmented=True, lanes=stats.refine_lanes,
                            windows=bool(windows))
        np.testing.assert_array_equal(levels[lo : lo + counts[i]].view(np.int64), want[3].view(np.int64))
        np.testing.assert_array_equal(iterations[lo : lo + counts[i]], want[4])
        eo += s.m
        lo += counts[i]
    # The copies give the same levels.
    n = sum(counts[: len(SIZES)])
    for c in range(1, copies):
        np.testing.assert_array_equal(levels[c * n : c * n + n].view(np.int64), levels[:n].view(np.int64))
