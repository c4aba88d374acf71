"""torch.autograd front end of the Numerov levels and their adjoint.

``numerov_levels(v, specs)`` solves the bound levels of a batch of tabulated
potentials on the GPU (scan + bracket + refine through libepseon_hip) and
returns them as a differentiable tensor.  Its backward is the adjoint kernel
``epseon_level_vjp``: for every converged level the eigenfunction is
recomputed on the device (two inward shots matched at min V) and

    dL/dV_i = sum_v dL/dE_v * psi_v(i)^2 * h,

the Hellmann-Feynman derivative of the discrete Numerov eigenproblem (exact
for the discretised problem).  Nothing of psi is stored between forward and
backward.

Chaining to potential parameters is ordinary torch autograd: tabulate V(theta)
(``morse_table`` does D_e (1 - exp(-a (r - r_e)))^2, in one kernel each way
where it can) on a grid that does not depend on theta, and backpropagate
through both.

The reference has no gradient path; its Python surface
(python/epseon_backend/device/gpu/_libepseon_gpu.pyi) and the algorithm record
(cpp/gpu/include/epseon/gpu/task_configurator/algorithm_config.hpp:75-199)
define the inputs this module takes: grid (min_r, max_r, point_count),
reduced mass from the two atom masses, the energy window below the asymptote
and the level range.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Sequence

import numpy as np
import torch

from . import capi


@dataclass
class LevelSpec:
    """Solver settings of one potential (grid, mass, window, levels)."""

    r_min: float
    r_max: float
    reduced_mass: float
    e_top: float
    n_energies: int
    level_min: int = 0
    level_count: int = 1


class LevelSolver:
    """A device context reused across calls (its arena and stream persist).

    Each forward loads the batch again; the backward of the most recent
    forward runs on the loaded state, an older one re-solves its saved V
    first (results are deterministic, so this only costs time)."""

    def __init__(self, device: int | torch.device | None = None, rel_tol: float = 1e-10,
                 max_iter: int = 200, refine_mode: int = capi.REFINE_AUTO) -> None:
        if device is None:
            device = torch.cuda.current_device()
        if isinstance(device, torch.device):
            device = device.index if device.index is not None else torch.cuda.current_device()
        self.device = int(device)
        self.rel_tol = float(rel_tol)
        self.max_iter = int(max_iter)
        self.ctx = capi.Context(self.device)
        self.ctx.set_refine_mode(refine_mode)
        self.generation = 0
        self.last_stats: capi.Stats | None = None

    def close(self) -> None:
        self.ctx.close()

    def _load_and_solve(self, v: torch.Tensor, specs: Sequence[LevelSpec]) -> None:
        """Upload the rows of v: straight from device memory when v lives on
        this solver's GPU, through the host otherwise."""
        rows, n = v.shape
        meta = [
            capi.Potential(values=range(n), r_min=s.r_min, r_max=s.r_max, reduced_mass=s.reduced_mass,
                           e_top=s.e_top, n_energies=s.n_energies, level_min=s.level_min,
                           level_count=s.level_count)
            for s in specs
        ]
        if v.is_cuda and v.device.index == self.device:
            vd = v.detach().to(torch.float64).contiguous()
            torch.cuda.current_stream(vd.device).synchronize()
            self.ctx.load_device(meta, vd.data_ptr(), [i * n for i in range(rows)])
        else:
            v_host = v.detach().to("cpu", torch.float64).contiguous().numpy()
            for i, m in enumerate(meta):
                m.values = v_host[i]
            self.ctx.load(meta)
        self.ctx.solve(self.rel_tol, self.max_iter)

    def solve(self, v: torch.Tensor, specs: Sequence[LevelSpec]) -> tuple[torch.Tensor, int]:
        """Levels of the rows of v (P, N) as a (P, L) float64 tensor on v's
        device, NaN where a level did not converge; plus the generation tag."""
        self._load_and_solve(v, specs)
        lv, st, _ = self.ctx.levels()
        lv = np.where(st == capi.LEVEL_OK, lv, np.nan)
        self.generation += 1
        counts = {s.level_count for s in specs}
        if len(counts) != 1:
            raise ValueError("numerov_levels needs the same level_count for every potential")
        out = torch.from_numpy(lv.reshape(len(specs), counts.pop())).to(v.device)
        return out, self.generation

    def vjp(self, v: torch.Tensor, specs: Sequence[LevelSpec], generation: int,
            grad_levels: torch.Tensor) -> torch.Tensor:
        """sum_l grad_levels[l] dE_l/dV as a tensor shaped like v."""
        if generation != self.generation:
            self._load_and_solve(v, specs)
            self.generation += 1
        g = torch.nan_to_num(grad_levels.detach().to(torch.float64), nan=0.0, posinf=0.0, neginf=0.0)
        if v.is_cuda:
            g = g.to(v.device).contiguous()
            out = torch.empty(v.shape[0] * v.shape[1], dtype=torch.float64, device=v.device)
            torch.cuda.current_stream(v.device).synchronize()
            self.ctx.level_vjp_device(g.data_ptr(), out.data_ptr())
        else:
            out = torch.from_numpy(self.ctx.level_vjp(g.reshape(-1).cpu().numpy()))
        self.last_stats = self.ctx.stats()
        return out.reshape(v.shape)


class _NumerovLevels(torch.autograd.Function):
    @staticmethod
    def forward(ctx, v: torch.Tensor, solver: LevelSolver, specs: tuple[LevelSpec, ...]) -> torch.Tensor:
        levels, gen = solver.solve(v, specs)
        ctx.solver = solver
        ctx.specs = specs
        ctx.generation = gen
        ctx.save_for_backward(v)
        return levels

    @staticmethod
    def backward(ctx, grad_levels: torch.Tensor):
        (v,) = ctx.saved_tensors
        grad_v = ctx.solver.vjp(v, ctx.specs, ctx.generation, grad_levels.reshape(-1))
        return grad_v.to(v.dtype), None, None


def numerov_levels(v: torch.Tensor, specs: Sequence[LevelSpec] | LevelSpec,
                   solver: LevelSolver | None = None) -> torch.Tensor:
    """Bound levels (P, L) of the potentials v (P, N) (cm^-1 on uniform grids),
    differentiable with respect to v through the adjoint kernel."""
    if v.dim() != 2:
        raise ValueError("v must be a (potentials, points) tensor")
    if isinstance(specs, LevelSpec):
        specs = [specs] * v.shape[0]
    if len(specs) != v.shape[0]:
        raise ValueError("one LevelSpec per potential is needed")
    if solver is None:
        solver = LevelSolver(v.device if v.is_cuda else None)
    return _NumerovLevels.apply(v, solver, tuple(specs))


def uniform_grid(r_min: torch.Tensor, r_max: torch.Tensor, n: int) -> torch.Tensor:
    """r_i = r_min + i h, h = (r_max - r_min)/(n - 1), for each potential (P, n)."""
    i = torch.arange(n, dtype=torch.float64, device=r_min.device)
    h = (r_max - r_min) / (n - 1)
    return r_min[:, None] + i[None, :] * h[:, None]


def _plain_tensor(t: torch.Tensor) -> bool:
    """Whether t's memory holds its values: an ordinary dense tensor, not a
    batched, negated or zero one.  False where torch lacks one of the private
    queries that tell."""
    if type(t) is not torch.Tensor and type(t) is not torch.nn.Parameter:
        return False
    try:
        wrapped = torch._C._functorch
        return (t.layout is torch.strided and not t.is_neg() and not t._is_zerotensor()
                and not wrapped.is_functorch_wrapped_tensor(t) and not wrapped.is_legacy_batchedtensor(t))
    except AttributeError:
        return False


def _eager() -> bool:
    """No tracer, transform, mode or forward-mode level is active: they see
    tensor operations, not a kernel.  False where torch lacks one of the
    private queries."""
    try:
        return not (torch.compiler.is_compiling() or torch.jit.is_tracing()
                    or torch._C._are_functorch_transforms_active()
                    or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack()
                    or torch.autograd.forward_ad._current_level >= 0)
    except AttributeError:
        return False


def _morse_kernel_takes(r: torch.Tensor, de: torch.Tensor, a: torch.Tensor, re: torch.Tensor) -> bool:
    """Whether the kernels of morse_kernels.hip compute this table: float64
    rows on one GPU without broadcasting, and gradients asked of all three
    parameters (then the tensors that are kept for the backward, and so must
    not change before it, are those that the tensor expressions keep) or of none.
    They are ahead at every size (forward and backward, 256 x 50,000 points:
    0.79 -> 0.09 ms; 7,001 points, where launches count: a fit step 1.00 -> 0.93 ms)."""
    if not (isinstance(r, torch.Tensor) and r.is_cuda and _eager() and r.dim() == 2 and r.is_contiguous()):
        return False
    for t in (r, de, a, re):
        if not (isinstance(t, torch.Tensor) and t.dtype is torch.float64 and t.device == r.device
                and _plain_tensor(t)):
            return False
    for t in (de, a, re):
        if t.dim() != 1 or t.shape[0] != r.shape[0]:
            return False
    if torch.is_grad_enabled():
        wanted = [t.requires_grad for t in (de, a, re)]
        if r.requires_grad or any(wanted) != all(wanted):
            return False
    return capi.load_library().epseon_morse_chunks(*r.shape) > 0


def _morse_forward(r: torch.Tensor, de: torch.Tensor, a: torch.Tensor, re: torch.Tensor,
                   v: torch.Tensor, d: torch.Tensor | None) -> None:
    de, a, re = de.contiguous(), a.contiguous(), re.contiguous()
    with torch.cuda.device(r.device):
        capi._check(capi.load_library().epseon_morse_table(
            r.data_ptr(), de.data_ptr(), a.data_ptr(), re.data_ptr(), r.shape[0], r.shape[1], v.data_ptr(),
            None if d is None else d.data_ptr(), torch.cuda.current_stream().cuda_stream))


class _MorseTable(torch.autograd.Function):
    """V and d = r - r_e; d is an output so that derivatives of the backward
    reach r_e through it."""

    @staticmethod
    def forward(ctx, r: torch.Tensor, de: torch.Tensor, a: torch.Tensor, re: torch.Tensor):
        v, d = torch.empty_like(r), torch.empty_like(r)
        _morse_forward(r, de, a, re, v, d)
        ctx.save_for_backward(d, de, a)
        ctx.set_materialize_grads(False)
        return v, d

    @staticmethod
    def backward(ctx, g: torch.Tensor | None, g_d: torch.Tensor | None):
        d, de, a = ctx.saved_tensors
        # Saved-tensor hooks may return anything that the expressions take.
        if g is not None and g_d is None and not torch.is_grad_enabled() and _eager() and d.is_cuda \
                and d.dim() == 2 and g.shape == d.shape and de.shape == a.shape == d.shape[:1] \
                and all(_plain_tensor(t) and t.dtype is torch.float64 and t.device == d.device
                        for t in (g, d, de, a)):
            return (None, *_MorseTable.kernel_vjp(g, d, de, a))
        g_de = g_a = g_re = None
        if g is not None:
            e = torch.exp(-a[:, None] * d)
            x = 1.0 - e
            t = 2.0 * g * (de[:, None] * x) * e
            g_de, g_a, g_re = (g * x * x).sum(1), (t * d).sum(1), -(t * a[:, None]).sum(1)
        if g_d is not None:
            g_re = -g_d.sum(1) if g_re is None else g_re - g_d.sum(1)
        return None, g_de, g_a, g_re

    @staticmethod
    def kernel_vjp(g: torch.Tensor, d: torch.Tensor, de: torch.Tensor, a: torch.Tensor):
        lib = capi.load_library()
        rows, points = d.shape
        g, d, de, a = g.contiguous(), d.contiguous(), de.contiguous(), a.contiguous()
        chunks = lib.epseon_morse_chunks(rows, points)
        grad = torch.empty((3, rows), dtype=torch.float64, device=d.device)
        part = torch.empty(3 * rows * chunks if chunks > 1 else 0, dtype=torch.float64, device=d.device)
        with torch.cuda.device(d.device):
            capi._check(lib.epseon_morse_vjp(g.data_ptr(), d.data_ptr(), de.data_ptr(), a.data_ptr(), rows, points,
                                             part.data_ptr() or None, grad.data_ptr(),
                                             torch.cuda.current_stream().cuda_stream))
        return grad.unbind(0)


def morse_table(r: torch.Tensor, de: torch.Tensor, a: torch.Tensor, re: torch.Tensor) -> torch.Tensor:
    """V = D_e (1 - exp(-a (r - r_e)))^2 per row of r (parameters are (P,))."""
    if _morse_kernel_takes(r, de, a, re):
        if torch.is_grad_enabled() and de.requires_grad:
            return _MorseTable.apply(r, de, a, re)[0]
        v = torch.empty_like(r)
        _morse_forward(r, de, a, re, v, None)
        return v
    x = 1.0 - torch.exp(-a[:, None] * (r - re[:, None]))
    return de[:, None] * x * x
