"""Batches on both sides of the sizes from which wide blocks read segment
tables and the normalisation packs its wavefronts take the variant they should
(epseon_stats.paths), and both variants agree with the oracle."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import oracle
from epseon_backend_amd.workloads import MorseSpec
from tests.helpers import problem_from_spec

pytestmark = pytest.mark.gpu


def _log(msg):
    sys.stdout.write(msg + "\n")
    sys.stdout.flush()


def _potentials(specs, count):
    from epseon_backend_amd import capi

    return [capi.Potential(values=s.table(), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.mu, e_top=s.de,
                           n_energies=s.m, level_min=0, level_count=count) for s in specs]


@pytest.mark.parametrize("windows", [0, 1])
@pytest.mark.parametrize("points, tables", [(16_383, False), (16_384, True)])
@pytest.mark.parametrize("lanes", [128, 256])
def test_wide_tables_from_16384_points(lanes, points, tables, windows):
    from epseon_backend_amd import capi

    _log(f"case: {points} points, {lanes} lanes, windows {windows}")
    spec = MorseSpec(20.0, 20000.0, 1.7, 1.6, 1.0, 5.0, points, 300)
    with capi.Context(0) as ctx:
        t = ctx.tuning()
        t.refine_mode, t.windows, t.segmented_lanes = capi.REFINE_SEGMENTED, windows, lanes
        ctx.set_tuning(t)
        ctx.load(_potentials([spec], 12))
        assert ctx.potential_info(0).point_count == points
        ctx.solve(1e-10, 200)
        assert bool(ctx.stats().paths & capi.PATH_WIDE_TABLES) == tables
        levels, status, iterations = ctx.levels()
    assert np.all(status == 0)
    want = oracle.solve(problem_from_spec(spec), 0, 12, 1e-10, 200, segmented=True, lanes=lanes, windows=bool(windows))
    np.testing.assert_array_equal(levels.view(np.int64), want[3].view(np.int64))
    np.testing.assert_array_equal(iterations, want[4])


# 18,000 points are 94 segments: 6,144 tasks from 66 potentials on.  63 levels
# leave a wavefront too full for packing to take one away.
@pytest.mark.parametrize("potentials, levels, packed", [(48, 17, False), (80, 17, True), (80, 63, False)])
def test_packed_normalisation_from_6144_tasks(potentials, levels, packed):
    from epseon_backend_amd import capi

    _log(f"case: {potentials} x 18,000 points x {levels} levels")
    specs = [MorseSpec(90.0, 20000.0, 1.7, 1.6, 1.0, 5.0, 18_000 + 7 * i, 256) for i in range(potentials)]
    grads = np.random.default_rng(3).standard_normal((potentials, levels))
    with capi.Context(0) as ctx:
        ctx.load(_potentials(specs, levels))
        ctx.solve(1e-10, 200)
        assert ctx.stats().paths & capi.PATH_PACKED_PSI == 0
        lv, st = (a.reshape(potentials, levels) for a in ctx.levels()[:2])
        grad = ctx.level_vjp(grads.reshape(-1))
        assert bool(ctx.stats().paths & capi.PATH_PACKED_PSI) == packed
        at = np.cumsum([0] + ctx.point_counts)
        some = {k: ctx.wavefunctions(k) for k in (0, potentials // 2, potentials - 1)}
    assert np.all(st == 0)
    for k, psi in some.items():
        p = problem_from_spec(specs[k])
        want = oracle.level_vjp(p, lv[k], grads[k])
        np.testing.assert_allclose(grad[at[k]:at[k + 1]], want, rtol=0, atol=1e-11 * np.abs(want).max())
        for l in (0, levels // 2, levels - 1):
            want = oracle.eigenfunction(p, lv[k][l])
            np.testing.assert_allclose(psi[l], want, rtol=0, atol=1e-12 * np.abs(want).max())
