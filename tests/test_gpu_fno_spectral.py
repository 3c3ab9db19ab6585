"""The spectral path as one call against its single calls, which other tests hold to float64: the same
launches, so the same bits.  And the gradients' common buffer."""

import numpy as np
import pytest
import torch

from fno_emulation import EmulatedFNO
from wavefunctionsimpython_amd import _abi
from wavefunctionsimpython_amd.fno import FNO3d, dft_tables


@pytest.mark.gpu
@pytest.mark.parametrize("n,m,C", [(32, 12, 32), (10, 2, 1), (33, 16, 5), (64, 6, 40)])
def test_spectral_path(n, m, C):
    dev = torch.device("cuda:0")
    t = dft_tables(n, m)
    F2, F2t, G2, G2t = (_abi.fno_stage_table(a, dev) for a in (t["F2"], t["F2"].T, t["G2"], t["G2"].T))
    g = torch.Generator(device=dev).manual_seed(3)

    def u(size):
        return torch.randn(size, generator=g, device=dev, dtype=torch.float32)

    m2, m3, tm = m * m, m ** 3, 2 * m
    Rr, Ri, T = u(m3 * C * C), u(m3 * C * C), u(C * n * n * tm)
    xs = 2 * C * n * m2
    a, b = ([u(xs), u(2 * C * m3), u(2 * C * m3), u(xs), u(C * n * n * tm)] for _ in range(2))
    _abi.fno_spectral(F2, G2, Rr, Ri, T, *a, n, m, C)
    U, X, O, Y, Z = b
    _abi.fno_stage(F2, T, U, tm, 2 * n, m, C * n)
    _abi.fno_stage(F2, U, X, tm, 2 * n, m2, C)
    _abi.fno_modes(Rr, Ri, X, O, m3, C)
    _abi.fno_stage(G2, O, Y, 2 * n, tm, m2, C)
    _abi.fno_stage(G2, Y, Z, 2 * n, tm, m, C * n)
    for x, y in zip(a, b):
        assert torch.equal(x, y)

    gr = u(m3 * C * C)
    grads = [gr.clone(), gr.clone(), gr.clone(), gr.clone()]
    in_place = T.clone()
    Y1, O1, d1, U1 = u(xs), u(2 * C * m3), u(2 * C * m3), u(xs)
    _abi.fno_spectral_backward(G2t, F2t, Rr, Ri, X, in_place, Y1, O1, d1, U1, in_place, grads[0], grads[1], n, m, C)
    d2 = torch.empty_like(d1)
    _abi.fno_stage(G2t, T, Y, tm, 2 * n, m, C * n)
    _abi.fno_stage(G2t, Y, O, tm, 2 * n, m2, C)
    _abi.fno_modes_backward(Rr, Ri, X, O, d2, grads[2], grads[3], m3, C)
    _abi.fno_stage(F2t, d2, U, 2 * n, tm, m2, C)
    _abi.fno_stage(F2t, U, Z, 2 * n, tm, m, C * n)
    assert torch.equal(in_place, Z) and torch.equal(d1, d2)
    assert torch.equal(grads[0], grads[2]) and torch.equal(grads[1], grads[3])


@pytest.mark.gpu
def test_spectral_path_limits():
    dev = torch.device("cuda:0")
    t = dft_tables(32, 12)
    F2 = _abi.fno_stage_table(t["F2"], dev)
    G2 = _abi.fno_stage_table(t["G2"], dev)
    z = torch.zeros(32 * 32 * 24, device=dev)
    with pytest.raises(ValueError):
        _abi.fno_spectral(G2, F2, z, z, z, z, z, z, z, z, 32, 12, 1)      # tables exchanged
    with pytest.raises(ValueError):
        _abi.fno_spectral(F2, G2, z, z, z[:-1], z, z, z, z, z, 32, 12, 1)  # T too short


def test_gradients_are_cleared_together():
    net = EmulatedFNO(8, width=5, modes=2, layers=2, in_channels=3, device=torch.device("cpu"))
    assert net._grad_all.is_contiguous()
    for k, g in net.grads.items():
        assert g.shape == net.params[k].shape and g.is_contiguous() and g.storage_offset() % 64 == 0
        g += 1.0
    own = torch.full_like(net.grads["Q"], 3.0)
    net.grads["Q"] = own
    net.zero_grad()
    assert all(np.all(g.numpy() == 0.0) for g in net.grads.values()) and net.grads["Q"] is own


def test_gradient_views_do_not_overlap():
    net = EmulatedFNO(8, width=5, modes=2, layers=1, in_channels=3, device=torch.device("cpu"))
    for i, g in enumerate(net.grads.values()):
        g.fill_(float(i + 1))
    assert all(np.all(g.numpy() == i + 1) for i, g in enumerate(net.grads.values()))
    assert isinstance(net, FNO3d)
