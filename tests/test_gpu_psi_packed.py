"""The normalisation with a potential's (segment, level) pairs packed into
wavefronts (batches of many eigenfunction tasks) against the one that gives
each segment its own: eigenfunctions and gradients are bit-identical, over
level counts around a wavefront's lanes, grids of every remainder of the
32-step block, unresolved potentials and levels that no bracket holds."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from epseon_backend_amd.workloads import MorseSpec

pytestmark = pytest.mark.gpu

LEVELS = [1, 2, 17, 31, 33, 41, 63, 64, 65, 70, 0, 129]


def _run(pots, grads):
    from epseon_backend_amd import capi

    with capi.Context(0) as ctx:
        ctx.load(pots)
        ctx.solve(1e-10, 200)
        levels, status, _ = (a.copy() for a in ctx.levels())
        grad = ctx.level_vjp(np.concatenate(grads))
        ctx.normalize()
        psi = [ctx.wavefunctions(k) for k in range(12)]
    return levels, status, grad, psi


def test_packed_pairs_match_single_segments():
    from epseon_backend_amd import capi

    sys.stdout.write("case: packed normalisation\n")
    sys.stdout.flush()
    rng = np.random.default_rng(11)
    pots, grads = [], []
    for i in range(156):
        # 18,000 points and more: 36 or more segments of 512 steps and a rest;
        # one in 13 does not resolve its window.
        n = 60 if i % 13 == 12 else 18_000 + 7 * i
        s = MorseSpec(60.0, 20000.0, 1.7, 1.6, 1.0, 5.0, n, 256)
        if n == 60:
            s = MorseSpec(50.0, 40000.0, 2.5, 2.0, 0.2, 9.0, n, 64)
        # The last three of a potential's levels may lie above its well.
        lmin = s.bound_levels() - 10 if i % 5 == 0 else 0
        c = LEVELS[i % len(LEVELS)]
        pots.append(capi.Potential(values=s.table(), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.mu, e_top=s.de,
                                   n_energies=s.m, level_min=lmin, level_count=c))
        grads.append(rng.standard_normal(c))
    part = 48
    levels, status, grad, psi = _run(pots, grads)
    levels1, status1, grad1, psi1 = _run(pots[:part], grads[:part])
    n_lv, n_pts = len(levels1), len(grad1)
    assert 0 < np.sum(status1 == 0) < n_lv
    np.testing.assert_array_equal(status[:n_lv], status1)
    np.testing.assert_array_equal(levels[:n_lv].view(np.int64), levels1.view(np.int64))
    np.testing.assert_array_equal(grad[:n_pts].view(np.int64), grad1.view(np.int64))
    assert np.all(np.isfinite(grad))
    for a, b in zip(psi, psi1):
        np.testing.assert_array_equal(a.view(np.int64), b.view(np.int64))
