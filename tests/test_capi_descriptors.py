"""The descriptor records that a load fills column by column, against the C
struct's layout and values."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from epseon_backend_amd import capi


def test_record_layout_is_the_struct():
    assert capi._DESC_DTYPE.itemsize == ctypes.sizeof(capi.PotentialDesc)
    for name, _ in capi.PotentialDesc._fields_:
        assert capi._DESC_DTYPE.fields[name][1] == getattr(capi.PotentialDesc, name).offset


@pytest.mark.parametrize("n", [0, 1, 2, 7])
def test_records_hold_the_potentials(n):
    pots = [capi.Potential(values=[0.0] * (4 + i), r_min=0.5 + i, r_max=9.0 + i, reduced_mass=1.5 + i, e_top=100.0 * i,
                           n_energies=np.int64(64 + i), level_min=i, level_count=2 * i) for i in range(n)]
    desc = capi._descriptors(pots, [len(p.values) for p in pots])
    structs = ctypes.cast(desc.ctypes.data, ctypes.POINTER(capi.PotentialDesc))
    assert len(desc) == max(n, 1)
    for i, p in enumerate(pots):
        assert structs[i].n_points == len(p.values)
        for name in ("r_min", "r_max", "reduced_mass", "e_top", "n_energies", "level_min", "level_count"):
            assert getattr(structs[i], name) == getattr(p, name)
    offsets = capi._offsets([len(p.values) for p in pots])
    assert offsets.tolist() == ([sum(4 + j for j in range(i)) for i in range(n)] or [0])
