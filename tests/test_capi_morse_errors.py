"""The Morse entry points leave their own message when they refuse a call."""
from __future__ import annotations

import pytest

from epseon_backend_amd import capi


@pytest.mark.parametrize("name", ["epseon_morse_table", "epseon_morse_vjp"])
@pytest.mark.parametrize("pointer, rows, points", [(None, 1, 1), (64, 0, 5), (64, 5, 0), (64, 1 << 23, 4096),
                                                   (64, -1, 3), (64, 1, 1 << 41)])
def test_a_refused_call_names_itself(name, pointer, rows, points):
    """No pointer is read: the sizes or the null pointers are refused first."""
    lib = capi.load_library()
    assert lib.epseon_scan(None) == capi.EPSEON_ERR_INVALID
    if pointer is not None:
        assert lib.epseon_morse_chunks(rows, points) == 0
    rc = getattr(lib, name)(pointer, pointer, pointer, pointer, rows, points, pointer, pointer, None)
    assert rc == capi.EPSEON_ERR_INVALID
    with pytest.raises(capi.EpseonError, match=name) as err:
        capi._check(rc)
    assert err.value.code == capi.EPSEON_ERR_INVALID
