"""A torch without one of the private queries that the Morse kernels' rule asks
takes the tensor expressions."""
from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

from epseon_backend_amd import autograd  # noqa: E402


def test_all_names_there():
    assert autograd._eager() and autograd._plain_tensor(torch.zeros(2))


@pytest.mark.parametrize("owner, name", [(torch._C, "_are_functorch_transforms_active"),
                                         (torch._C, "_len_torch_dispatch_stack"),
                                         (torch._C, "_len_torch_function_stack"),
                                         (torch.autograd.forward_ad, "_current_level"),
                                         (torch._C._functorch, "is_functorch_wrapped_tensor"),
                                         (torch._C._functorch, "is_legacy_batchedtensor")])
def test_a_missing_name_rules_the_kernels_out(monkeypatch, owner, name):
    monkeypatch.delattr(owner, name)
    assert not (autograd._eager() and autograd._plain_tensor(torch.zeros(2)))


def test_no_functorch_module(monkeypatch):
    monkeypatch.delattr(torch._C, "_functorch")
    assert not autograd._plain_tensor(torch.zeros(2))
