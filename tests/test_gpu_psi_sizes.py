"""Eigenfunctions and adjoint against the oracle where the segmented passes can
go wrong: both shots' lengths through every remainder of the 32-step block, at
and around a segment's length, and level counts around the lanes of a
wavefront.  Tolerances as in the full-size tests: the two sides run the same
recurrence from segment starts that differ by rounding."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import oracle
from epseon_backend_amd.workloads import K_CM

pytestmark = pytest.mark.gpu


def _problem(n, match, rng, levels):
    """A harmonic well of about `levels` bound levels with its minimum at
    `match` points from the left end."""
    i = np.arange(n) - match
    v = 4_000.0 * (i / max(match, n - 1 - match)) ** 2 + rng.uniform(0.0, 1.0)
    v[match] -= 1.0
    # Classical phase at the window top: about pi per level.
    h = 1.0 / (n - 1)
    theta = min(1.0, np.pi * levels / (0.6 * n))
    mu = theta * theta * K_CM / (h * h * 3_000.0)
    return oracle.Problem(v=v, r_min=0.0, r_max=1.0, mu=mu, e_top=float(v.min()) + 3_000.0, m=max(64, 8 * levels))


def _check(probs, counts):
    from epseon_backend_amd import capi

    with capi.Context(0) as ctx:
        ctx.load([capi.Potential(values=p.v, r_min=p.r_min, r_max=p.r_max, reduced_mass=p.mu, e_top=p.e_top,
                                 n_energies=p.m, level_min=0, level_count=c) for p, c in zip(probs, counts)])
        ctx.solve(1e-10, 200)
        lv, st, _ = ctx.levels()
        g = np.random.default_rng(5).standard_normal(len(lv))
        grad = ctx.level_vjp(g)
        every = ctx.all_wavefunctions()
    lo = o = found = 0
    for p, c, psi in zip(probs, counts, every):
        ok = st[lo:lo + c] == 0
        found += int(ok.sum())
        for l in range(c):
            if not ok[l]:
                assert np.all(psi[l] == 0.0)
                continue
            want = oracle.eigenfunction(p, lv[lo + l])
            np.testing.assert_allclose(psi[l], want, rtol=0, atol=1e-12 * np.abs(want).max(), err_msg=f"{p.n}/{l}")
        want = oracle.level_vjp(p, np.where(ok, lv[lo:lo + c], np.nan), g[lo:lo + c])
        np.testing.assert_allclose(grad[o:o + p.n], want, rtol=0, atol=1e-11 * max(np.abs(want).max(), 1e-300))
        lo += c
        o += p.n
    return found


def test_every_shot_remainder():
    rng = np.random.default_rng(1)
    probs = [_problem(n, m, rng, 2) for n, m in
             [(6 + 2 * k, 2 + k) for k in range(40)] + [(120, m) for m in range(40, 75)] +
             [(2 * s + 3, s) for s in (511, 512, 513, 1024, 1025)] + [(4000, 700), (4000, 3300)]]
    sys.stdout.write(f"case: {len(probs)} grids\n")
    sys.stdout.flush()
    assert _check(probs, [2] * len(probs)) >= len(probs)


@pytest.mark.parametrize("levels", [1, 31, 32, 33, 63, 64, 65, 129, 300])
def test_level_counts_around_a_wavefront(levels):
    rng = np.random.default_rng(2)
    sys.stdout.write(f"case: {levels} levels\n")
    sys.stdout.flush()
    probs = [_problem(2_500, 1_100, rng, levels), _problem(3_001, 1_700, rng, levels)]
    assert _check(probs, [levels, levels]) >= levels
