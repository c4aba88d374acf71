"""Scans on both sides of the limits up to which they run in spread workgroups
(wavefronts per SIMD, of even and of ragged shots) are the oracle's bit for bit."""
from __future__ import annotations

import dataclasses
import sys

import numpy as np
import pytest

from epseon_backend_amd import capi
from epseon_backend_amd.workloads import MorseSpec
from tests.helpers import problem_from_spec

pytestmark = pytest.mark.gpu


# 64 wavefronts per potential: 30, 38 and 50 per SIMD of 1,024, whole grids.
@pytest.mark.parametrize("longest", [300, 3_000])
@pytest.mark.parametrize("count", [480, 608, 800])
def test_scan_matches_oracle(count, longest):
    sys.stdout.write(f"case: {count} potentials, longest {longest}\n")
    sys.stdout.flush()
    base = MorseSpec(1.0, 20000.0, 1.7, 1.6, 1.0, 5.0, 300, 4_090)
    specs = [dataclasses.replace(base, mu=1.0 + 0.001 * i, n=longest if i == 17 else 300 - i % 7) for i in range(count)]
    with capi.Context(0) as ctx:
        t = ctx.tuning()
        t.windows = 0
        ctx.set_tuning(t)
        ctx.load([capi.Potential(values=s.table(), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.mu, e_top=s.de,
                                 n_energies=s.m, level_min=0, level_count=1) for s in specs])
        ctx.scan()
        got = [np.array(x).reshape(count, base.m) for x in ctx.scan_results()]
        assert all(ctx.potential_info(p).flags == 0 for p in range(count))
    for p in (0, 17, count // 2, count - 1):
        for x, want in zip(got, problem_from_spec(specs[p]).scan(False)):
            np.testing.assert_array_equal(x[p], want)
