"""Gradients of the network that the caller takes out or puts in (host logic, on the CPU)."""

import torch

from wavefunctionsimpython_amd.fno import FNO3d


def _net():
    net = FNO3d(8, width=4, modes=2, layers=2, device=torch.device("cpu"))
    for g in net.grads.values():
        g.fill_(1.0)
    return net


def test_zero_grad_clears_every_gradient():
    net = _net()
    net.zero_grad()
    assert all(not g.any() for g in net.grads.values())


def test_zero_grad_leaves_a_gradient_that_the_caller_took_out():
    net = _net()
    taken = net.grads["W0"]
    net.grads["W0"] = torch.full_like(taken, 2.0)
    net.zero_grad()
    assert bool((taken == 1.0).all())
    assert all(not g.any() for g in net.grads.values())


def test_zero_grad_with_all_gradients_replaced():
    net = _net()
    taken = net.grads
    net.grads = {k: torch.full_like(g, 2.0) for k, g in taken.items()}
    net.zero_grad()
    assert all(bool((g == 1.0).all()) for g in taken.values())
    assert all(not g.any() for g in net.grads.values())
