"""A potential's eigenfunctions and gradient have the same bits whatever else
was loaded with it, and the allocation-free adjoint goes through batches whose
segments exceed its scratch in parts."""
from __future__ import annotations

import sys

import numpy as np
import pytest

from epseon_backend_amd.workloads import batched, differentiation

pytestmark = pytest.mark.gpu


def _log(msg):
    sys.stdout.write(msg + "\n")
    sys.stdout.flush()


def _potentials(specs, counts, m=256):
    from epseon_backend_amd import capi

    return [capi.Potential(values=s.table(), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.mu, e_top=s.de,
                           n_energies=m, level_min=0, level_count=c) for s, c in zip(specs, counts)]


def _run(pots, grads):
    """(levels, gradients, eigenfunctions), split by potential."""
    import torch

    from epseon_backend_amd import capi

    with capi.Context(0) as ctx:
        # One refinement arithmetic for every batch size.
        t = ctx.tuning()
        t.refine_mode, t.segmented_lanes, t.windows = capi.REFINE_SEGMENTED, 64, 1
        ctx.set_tuning(t)
        ctx.load(pots)
        ctx.solve(1e-10, 200)
        levels = ctx.levels()[0].copy()
        g = torch.from_numpy(np.concatenate(grads)).cuda()
        out = torch.full((ctx.v_span,), float("nan"), dtype=torch.float64, device="cuda")
        ctx.level_vjp_noalloc(g.data_ptr(), out.data_ptr())
        grad = out.cpu().numpy()
        psi = [ctx.wavefunctions(k) for k in range(len(pots))]
    at = np.cumsum([0] + [p.level_count for p in pots])
    pt = np.cumsum([0] + [len(p.values) for p in pots])
    return [(levels[at[k]:at[k + 1]], grad[pt[k]:pt[k + 1]], psi[k]) for k in range(len(pots))]


# Between them the batches hold from a few to some thousand segments of any
# length that a potential's size could give.
@pytest.mark.parametrize("points, count, levels", [(2_500, 300, 24), (64_000, 16, 20), (200_001, 5, 70)])
def test_bits_do_not_depend_on_the_batch(points, count, levels):
    _log(f"case: {count} x {points} points x {levels} levels, whole and one by one")
    specs = batched(count)
    for i, s in enumerate(specs):
        s.n = points + 3 * i
    counts = [levels + i % 3 for i in range(count)]
    rng = np.random.default_rng(4)
    grads = [rng.standard_normal(c) for c in counts]
    pots = _potentials(specs, counts)
    whole = _run(pots, grads)
    for k in (0, count // 2, count - 1):
        _log(f"potential {k}")
        alone = _run(pots[k:k + 1], grads[k:k + 1])[0]
        assert np.sum(np.isfinite(alone[0])) > 0
        for a, b in zip(whole[k], alone):
            np.testing.assert_array_equal(a.view(np.int64), b.view(np.int64))


def test_group_size_with_many_segments():
    """Tasks of one group and of groups of one through the drop-in module."""
    from epseon_backend_amd.device.gpu import _libepseon_gpu as m

    interface = m.EpseonComputeContext.create().get_device_interface(0)
    specs = differentiation(12, n_points=50_000)
    cfgs = [m.MorsePotentialConfig(dissociation_energy=s.de, equilibrium_bond_distance=s.re, well_width=s.a,
                                   min_r=s.r_min, max_r=s.r_max, point_count=s.n) for s in specs]
    out = []
    for group in (1, 12):
        _log(f"case: 12 x 50,000 points, group_size {group}")
        c = (
            interface.get_task_configurator("float64")
            .set_hardware_config(potential_buffer_size=64000, group_size=group, allocation_block_size=1 << 24)
            .set_morse_potential_batch(cfgs)
            .set_vibwa_algorithm(mass_atom_0=1.0, mass_atom_1=1.0, integration_step=0.1,
                                 min_distance_to_asymptote=0.0, min_level=0, max_level=15)
            .set_reduced_masses([s.mu for s in specs])
            .set_trial_energy_counts([256] * len(specs))
            .set_eigenfunction_output(True)
        )
        handle = interface.submit_task(c)
        handle.wait()
        out.append((handle.get_levels().copy(), [x.copy() for x in handle.get_wavefunctions()]))
    np.testing.assert_array_equal(out[0][0].view(np.int64), out[1][0].view(np.int64))
    for a, b in zip(out[0][1], out[1][1]):
        np.testing.assert_array_equal(a.view(np.int64), b.view(np.int64))


# 256 potentials of 2,000 points: about 30 MB of maps and checkpoints in
# segments of 512 steps, and 120 MB, twice the scratch, in their own.  Two of
# 50,000 points around the number of pairs from which segments stay long.
@pytest.mark.parametrize("points, counts", [(2_000, [(40, 100, 170, 300, 700)[i % 5] for i in range(256)]),
                                            (50_000, [1_100, 900])])
def test_noalloc_in_parts_equals_level_vjp(points, counts):
    import torch

    from epseon_backend_amd import capi

    _log(f"case: {len(counts)} x {points} points, {min(counts)} to {max(counts)} levels")
    specs = differentiation(len(counts), n_points=points)
    with capi.Context(0) as ctx:
        ctx.load(_potentials(specs, counts))
        ctx.solve(1e-10, 200)
        g = torch.from_numpy(np.random.default_rng(6).standard_normal(sum(counts))).cuda()
        want = torch.full((ctx.v_span,), float("nan"), dtype=torch.float64, device="cuda")
        ctx.level_vjp_device(g.data_ptr(), want.data_ptr())
        for _ in range(2):
            got = torch.full_like(want, float("nan"))
            ctx.level_vjp_noalloc(g.data_ptr(), got.data_ptr())
            np.testing.assert_array_equal(got.cpu().numpy().view(np.int64), want.cpu().numpy().view(np.int64))
        assert torch.isfinite(want).all() and want.abs().max() > 0.0
