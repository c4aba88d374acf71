"""Morse table kernels against the tensor expressions on the CPU.

Bounds, u = 2^-53: the exponentials of the two sides differ by 2 ulp of e at
most, so y = 1 - e by 4 u e and its own rounding, and a term of V or of a
gradient by at most 32 u of the same term with |y| + e in the place of y; a
sum of n terms adds n u of the sum of their magnitudes.
"""
from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

from epseon_backend_amd import autograd  # noqa: E402

pytestmark = pytest.mark.gpu

U = 2.0**-53


def _inputs(rows, n, seed=0):
    gen = torch.Generator().manual_seed(seed)
    rand = lambda *s: torch.rand(*s, generator=gen, dtype=torch.float64)  # noqa: E731
    r = 0.4 + torch.cumsum(rand(rows, n), 1) * (8.0 / n)
    return r, 1e4 + 1e4 * rand(rows), 1.0 + rand(rows), 0.7 + rand(rows), rand(rows, n) - 0.5


def _table(r, theta, dev):
    p = [t.to(dev).requires_grad_() for t in theta]
    return p, autograd.morse_table(r.to(dev), *p)


@pytest.mark.parametrize("rows,n", [(1, 1), (3, 2), (5, 255), (2, 256), (3, 257), (1, 2047), (4, 2048), (3, 2049),
                                    (1, 4097), (2, 7001), (300, 33), (1, 600_001)])
def test_table_and_gradient(rows, n):
    r, de, a, re, g = _inputs(rows, n)
    assert autograd._morse_kernel_takes(*(t.cuda() for t in (r, de, a, re)))
    p, v = _table(r, (de, a, re), "cuda")
    plain = autograd.morse_table(r.cuda(), *(t.cuda() for t in (de, a, re)))
    assert torch.equal(plain, v.detach())
    q, w = _table(r, (de, a, re), "cpu")
    d = r - re[:, None]
    e = torch.exp(-a[:, None] * d)
    m = (1.0 - e).abs() + e
    assert ((v.detach().cpu() - w.detach()).abs() <= 32 * U * de[:, None] * m * m).all()
    got = torch.autograd.grad(v, p, g.cuda(), retain_graph=True)
    again = torch.autograd.grad(v, p, g.cuda().t().contiguous().t())
    want = torch.autograd.grad(w, q, g)
    h = 2.0 * g.abs() * de[:, None] * m * e
    for x, y, z, s in zip(got, again, want, (g.abs() * m * m, h * d.abs(), h * a[:, None])):
        assert torch.equal(x, y)
        assert ((x.cpu() - z).abs() <= (32 + n) * U * s.sum(1)).all()


def test_further_derivatives_transforms_and_changed_inputs():
    r, de, a, re, g = _inputs(3, 9)
    theta = (de * 1e-4, a, re)
    second = []
    for dev in ("cuda", "cpu"):
        p, v = _table(r, theta, dev)
        first = torch.autograd.grad(v, p, g.to(dev), create_graph=True)
        second.append(torch.autograd.grad(sum((t * t).sum() for t in first), p, retain_graph=True))
        batched = torch.autograd.grad(v, p, torch.stack([g, 2 * g]).to(dev), is_grads_batched=True)
        for t, b in zip(first, batched):
            torch.testing.assert_close(b, torch.stack([t, 2 * t]).detach(), rtol=1e-12, atol=1e-12)
    for x, y in zip(*second):
        torch.testing.assert_close(x.cpu(), y, rtol=1e-11, atol=1e-11)
    # Forward mode and vmap see the tensor expressions.
    cuda = [t.cuda() for t in (r, *theta)]
    jac = [f(autograd.morse_table, argnums=2)(*cuda) for f in (torch.func.jacfwd, torch.func.jacrev)]
    torch.testing.assert_close(jac[0], jac[1], rtol=1e-12, atol=1e-12)
    # r and r_e may change between the passes; a may not.
    p = [t.clone().requires_grad_() for t in cuda[1:]]
    grid = cuda[0].clone()
    v = autograd.morse_table(grid, *p)
    want = torch.autograd.grad(v, p, g.cuda(), retain_graph=True)
    with torch.no_grad():
        grid.zero_()
        p[2].zero_()
    for x, y in zip(torch.autograd.grad(v, p, g.cuda(), retain_graph=True), want):
        assert torch.equal(x, y)
    # Hooks may hand back other types.
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t.float(), lambda t: t):
        u = autograd.morse_table(cuda[0], *p[:2], cuda[3].clone().requires_grad_())
    assert torch.isfinite(torch.autograd.grad(u, p[0], g.cuda())[0]).all()
    with torch.no_grad():
        p[1].zero_()
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(v, p, g.cuda())


@pytest.mark.parametrize("change", ["r_grad", "some", "broadcast", "strided", "float32"])
def test_other_forms_take_the_tensor_expressions(change):
    r, de, a, re, _ = (t.cuda() for t in _inputs(4, 6))
    if change == "r_grad":
        r.requires_grad_()
    elif change == "some":
        a.requires_grad_()
    elif change == "broadcast":
        r = r[:1]
    elif change == "strided":
        r = r[:, ::2]
    else:
        r = r.float()
    assert not autograd._morse_kernel_takes(r, de, a, re)
    x = 1.0 - torch.exp(-a[:, None] * (r - re[:, None]))
    assert torch.equal(autograd.morse_table(r, de, a, re), de[:, None] * x * x)
