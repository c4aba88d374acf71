"""The refinement's statistics are those of the batch that is loaded, also of
one that asks for no levels."""
from __future__ import annotations

import sys

import pytest

from epseon_backend_amd.workloads import batched

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("separate", [False, True])
def test_a_batch_without_levels_after_one_with(separate):
    from epseon_backend_amd import capi

    sys.stdout.write(f"case: separate {separate}\n")
    sys.stdout.flush()
    converged = []
    with capi.Context(0) as ctx:
        for count in (5, 0, 3):
            ctx.load([capi.Potential(values=s.table(), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.mu, e_top=s.de,
                                     n_energies=s.m, level_min=0, level_count=count) for s in batched(2)])
            if separate:
                ctx.scan()
                ctx.refine(1e-10, 200)
            else:
                ctx.solve(1e-10, 200)
            stats = ctx.stats()
            converged.append(stats.levels_converged)
            assert (stats.refine_point_updates > 0) == (count > 0)
    assert converged == [10, 0, 6]
