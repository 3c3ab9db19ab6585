"""complex128 split step as two launches (kernel class yz_split) against the passes and the oracle."""

import numpy as np
import pytest
import torch

import oracle
from wavefunctionsimpython_amd import _abi

pytestmark = pytest.mark.gpu

DX, DT = (0.4, 0.35, 0.3), 0.01
C128 = _abi.WFS_C128


def _plan(shape, split, batch=1):
    p = _abi.Plan(shape, DX, DT, 1.0, C128, _abi.WFS_METHOD_FOURIER, batch=batch)
    p.set_variant("yz_split", split)
    return p


def _state(shape, dev, seed=0):
    rng = np.random.default_rng(seed)
    psi = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    V = rng.uniform(-0.5, 0.5, shape) - 0.05j * rng.random(shape)
    V[..., shape[-3] // 2:, :, :] = V[..., shape[-3] // 2:shape[-3] // 2 + 1, :, :]    # equal x planes
    return torch.from_numpy(psi).to(dev), torch.from_numpy(V.astype(np.complex64)).to(dev)


@pytest.mark.parametrize("n", [64, 96, 128, 192])
@pytest.mark.parametrize("nx,steps", [(8, 1), (32, 3), (96, 2), (256, 2)])
def test_split_matches_passes(dev, n, nx, steps):
    shape = (nx, n, n)
    psi, V = _state(shape, dev, n + nx)
    out = []
    for split in (0, 1):
        p = _plan(shape, split)
        a = psi.clone()
        p.step(a, V, steps)            # table of the call
        p.step(a, None, 1)             # table kept
        out.append(a)
    torch.cuda.synchronize()
    assert oracle.relative_l2(out[1].cpu().numpy(), out[0].cpu().numpy()) < 1e-13


def test_split_matches_oracle_and_follows_the_potential(dev):
    shape = (16, 64, 64)
    psi, V = _state(shape, dev, 3)
    p = _plan(shape, 1)
    a = psi.clone()
    p.set_potential(V)
    p.step(a, None, 2)
    W = V.clone()
    W[5:7] *= 0.5
    p.set_potential_planes(W, 5, 7)
    p.step(a, None, 2)
    p.set_variant("yz_split", 0)       # the table moves to the passes' order and back
    p.step(a, None, 1)
    p.set_variant("yz_split", 1)
    p.step(a, None, 1)
    ref = oracle.split_step(psi.cpu().numpy(), V.cpu().numpy(), DX, DT, 1.0, nsteps=2)
    ref = oracle.split_step(ref, W.cpu().numpy(), DX, DT, 1.0, nsteps=4)
    assert oracle.relative_l2(a.cpu().numpy(), ref) < 1e-12


@pytest.mark.parametrize("n", [64, 96, 128])
def test_split_packets_equal_single_runs(dev, n):
    shape, batch = (16, n, n), 3
    rng = np.random.default_rng(n)
    axes = [rng.uniform(-1, 1, (batch, m)) for m in shape]
    psi = _state((batch,) + shape, dev, n)[0]
    p = _plan(shape, 1, batch)
    p.set_potential_axes(*axes)
    a = psi.clone()
    p.step(a, None, 3)
    for i in range(batch):
        q = _plan(shape, 1)
        q.set_potential_axes(*(x[i] for x in axes))
        b = psi[i].clone()
        q.step(b, None, 3)
        assert torch.equal(a[i], b)


def test_split_defaults_and_switches(dev):
    def on(shape, precision=C128):
        return _abi.Plan(shape, DX, DT, 1.0, precision, _abi.WFS_METHOD_FOURIER).variants()["yz_split"]
    assert on((64, 64, 64)) and on((8, 96, 96)) and on((256, 192, 192))
    assert not (on((192, 64, 64)) or on((512, 96, 96)) or on((32, 32, 32)) or on((64, 128, 96)) or on((8, 256, 256)))
    assert not on((64, 64, 64), _abi.WFS_C64)
    p = _abi.Plan((16, 64, 64), DX, DT, 1.0, C128, _abi.WFS_METHOD_FOURIER)
    p.set_variant("yz_plane", 1)
    assert p.variants()["yz_split"] == 0
    with pytest.raises(_abi.WfsError):
        _abi.Plan((16, 32, 32), DX, DT, 1.0, C128, _abi.WFS_METHOD_FOURIER).set_variant("yz_split", 1)
