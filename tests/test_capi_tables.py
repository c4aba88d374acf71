"""The host buffer that Context.load gathers the tables in: kept for the next
load up to a bound, given back above it, and one load's alone while it runs."""
from __future__ import annotations

import ctypes

import numpy as np

from epseon_backend_amd import capi


class _Library:
    """Stands in for the C library: records the tables of each load."""

    def __init__(self):
        self.loads, self.during = [], None

    def epseon_load_potentials(self, handle, count, desc, v, offsets):
        during, self.during = self.during, None
        if during is not None:
            during()
        total = sum(desc[i].n_points for i in range(count))
        self.loads.append(np.ctypeslib.as_array(ctypes.cast(v, ctypes.POINTER(ctypes.c_double)), (total,))[:1000].copy())
        return capi.EPSEON_OK


def _context():
    ctx = object.__new__(capi.Context)
    ctx._lib, ctx._h = _Library(), ctypes.c_void_p()
    ctx._tables = np.empty(1)
    return ctx


def _batch(*values):
    return [capi.Potential(values=v, r_min=0.0, r_max=1.0, reduced_mass=1.0, e_top=1.0, n_energies=4) for v in values]


def test_a_large_buffer_is_given_back():
    ctx = _context()
    ctx.load(_batch(np.zeros(20_000), np.ones(5)))
    kept = ctx._tables
    assert len(kept) == 20_005
    ctx.load(_batch(np.full(7, 3.0)))
    assert ctx._tables is kept
    np.testing.assert_array_equal(ctx._lib.loads[1], np.full(7, 3.0))
    ctx.load(_batch(np.zeros((256 << 17) + 1)))
    assert ctx._tables.nbytes < 1000
    assert ctx.point_counts == [(256 << 17) + 1]


def test_a_load_during_another_leaves_its_tables_alone():
    ctx = _context()
    ctx.load(_batch(np.zeros(100)))
    ctx._lib.during = lambda: ctx.load(_batch(np.full(50, 2.0)))
    ctx.load(_batch(np.full(60, 1.0), np.full(40, 4.0)))
    np.testing.assert_array_equal(ctx._lib.loads[1], np.full(50, 2.0))
    np.testing.assert_array_equal(ctx._lib.loads[2], np.r_[np.full(60, 1.0), np.full(40, 4.0)])
