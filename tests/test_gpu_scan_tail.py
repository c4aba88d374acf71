"""Scan shots of every remainder: grids whose step count leaves 0 to 31 steps
after the last 32-step super-block, none to three super-blocks after the last
128-step iteration, and that end inside, at or past the first lines the shot
touches ahead of itself, for every node-sampling stride, bit-exact against the
oracle."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import oracle
from epseon_backend_amd.workloads import K_CM, MorseSpec
from tests.helpers import problem_from_spec

pytestmark = pytest.mark.gpu

# Steps (points - 2): every remainder below 32 once, 128-step iterations with
# 0 to 3 super-blocks left, and both sides of 1024 points and twice that.
STEPS = sorted(set(range(2, 34)) | {47, 48, 49, 63, 64, 65, 95, 96, 97, 127, 128, 129, 160, 191, 192, 255, 256, 257,
                                    1020, 1022, 1023, 1024, 1025, 1040, 1151, 1152, 1153, 1279, 2047, 2048, 2050, 4095})


@pytest.mark.parametrize("stride", [1, 2, 4, 8, 16, 32])
def test_scan_remainders_match_oracle(stride):
    from epseon_backend_amd import capi

    sys.stdout.write(f"case: stride {stride}, {len(STEPS)} grids\n")
    sys.stdout.flush()
    # The phase per step at the window top, 1.2 strides short of pi/2 per
    # sample, fixes the mass.
    de, a, re, span = 20000.0, 1.0, 1.2, 0.8
    theta = 0.5 * np.pi / (1.2 * stride)
    specs = []
    for steps in STEPS:
        h = span / (steps + 1)
        mu = theta * theta * K_CM / (h * h * de)
        specs.append(MorseSpec(mu, de, a, re, re - 0.35, re - 0.35 + span, steps + 2, 70))
    with capi.Context(0) as ctx:
        t = ctx.tuning()
        t.windows = 0
        ctx.set_tuning(t)
        ctx.load([capi.Potential(values=s.table(), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.mu, e_top=s.de,
                                 n_energies=s.m, level_min=0, level_count=0) for s in specs])
        ctx.scan()
        nodes, far, resc = ctx.scan_results()
        infos = [ctx.potential_info(i) for i in range(len(specs))]
    for i, s in enumerate(specs):
        prob = problem_from_spec(s)
        assert prob.usable and infos[i].flags == 0
        assert infos[i].stride == stride and infos[i].point_count == s.n
        want = oracle.solve(prob, 0, 0, windows=False)[:3]
        at = slice(70 * i, 70 * (i + 1))
        np.testing.assert_array_equal(nodes[at], want[0])
        np.testing.assert_array_equal(resc[at], want[2])
        np.testing.assert_array_equal(far[at].view(np.int64), np.asarray(want[1]).view(np.int64))
