"""The load passes (table statistics, walls, band windows) against the oracle
at the sizes where they can go wrong: tables around the chunk length and its
multiples, walls and minima at the ends and on chunk borders, fringes that end
inside one walk step, after several, or at the grid's end, and both walk widths
(below and from 64 potentials)."""
from __future__ import annotations

import sys

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

CHUNK = 4096  # a multiple of both chunk lengths
SIZES = [4, 5, 63, 64, 65, 255, 257, 1023, 1024, 1025, CHUNK - 1, CHUNK, CHUNK + 1, 2 * CHUNK, 2 * CHUNK + 7, 40_001, 300_007]


def _table(rng, n, kind):
    """A well with its minimum at the left end, the right end, a chunk border
    or inside, and walls steep enough to be trimmed or not."""
    at = {"left": 0, "right": n - 1, "border": min(n - 1, CHUNK - 1), "inside": n // 3}[kind[0]]
    x = (np.arange(n) - at) / n
    v = 30_000.0 * x * x + 25.0 * rng.standard_normal(n)
    if kind[1] == "walls":
        v = v + 1e9 * np.maximum(0.0, np.abs(x) - 0.4) ** 2
    return v


@pytest.mark.parametrize("copies", [1, 5])
def test_windows_and_trim_match_oracle(copies):
    import torch

    from epseon_backend_amd import capi

    rng = np.random.default_rng(20261205)
    kinds = [("left", "flat"), ("right", "walls"), ("border", "walls"), ("inside", "flat"), ("inside", "walls")]
    probs = []
    for i, n in enumerate(SIZES * copies):
        v = _table(rng, n, kinds[i % len(kinds)])
        # beta (E_top - V_min) near 1e-3, so walls from V_min + 5e5 on.
        h = oracle.grid_step(0.0, 1.0, n)
        mu = 12.0 * 16.857629191640175 * 1e-6 / (h * h)
        probs.append(oracle.Problem(v=v, r_min=0.0, r_max=1.0, mu=mu, e_top=float(v.min()) + 2000.0, m=16))
    sys.stdout.write(f"case: {len(probs)} tables\n")
    sys.stdout.flush()
    pots = [capi.Potential(values=p.v, r_min=p.r_min, r_max=p.r_max, reduced_mass=p.mu, e_top=p.e_top,
                           n_energies=p.m, level_min=0, level_count=0) for p in probs]
    flat = torch.from_numpy(np.concatenate([p.v for p in probs])).cuda()
    offsets = np.concatenate([[0], np.cumsum([len(p.v) for p in probs])])[:-1]
    torch.cuda.synchronize()
    with capi.Context(0) as ctx:
        t = ctx.tuning()
        t.windows = 1
        ctx.set_tuning(t)
        for load in ("host", "device"):
            if load == "host":
                ctx.load(pots)
            else:
                ctx.load_device(pots, flat.data_ptr(), [int(o) for o in offsets])
            for i, p in enumerate(probs):
                info = ctx.potential_info(i)
                b = oracle.beta(oracle.grid_step(p.r_min, p.r_max, len(p.v)), p.mu)
                first, last, usable = oracle.trim(p.v, b, p.e_top)
                assert (info.flags == 0) == usable
                if not usable:
                    continue
                assert (info.first_point, info.point_count) == (first, last - first + 1)
                assert info.e_lo == p.v.min()
                uv = oracle.scaled_potential(p.v[first:last + 1], b)
                want = oracle.band_windows(uv, b, float(p.v.min()), p.e_top)
                lo, hi, _ = ctx.band_windows(i)
                np.testing.assert_array_equal(lo, want[:, 0])
                np.testing.assert_array_equal(hi, want[:, 1])


@pytest.mark.parametrize("n", [CHUNK - 1, CHUNK + 3, 3 * CHUNK + 1])
def test_first_bad_value_is_named(n):
    import torch

    from epseon_backend_amd import capi

    v = np.linspace(-1.0, 1.0, n) ** 2 * 1e4
    with capi.Context(0) as ctx:
        for at in (0, n // 2, n - 1):
            w = v.copy()
            w[at] = np.nan
            w[min(n - 1, at + 300)] = np.inf
            t = torch.from_numpy(w).cuda()
            torch.cuda.synchronize()
            pot = capi.Potential(values=w, r_min=0.0, r_max=1.0, reduced_mass=1.0, e_top=5e3, n_energies=4,
                                 level_min=0, level_count=0)
            for load in (lambda: ctx.load([pot]), lambda: ctx.load_device([pot], t.data_ptr(), [0])):
                with pytest.raises(capi.EpseonError, match=rf"V\[{at}\] is not finite"):
                    load()
