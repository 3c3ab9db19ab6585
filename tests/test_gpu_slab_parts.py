"""The slab y-z launch that exchanges real and imaginary parts in turn (more row groups than CUs) against
the launch that exchanges whole values (one group per CU): the same bits, and the oracle's result."""

import numpy as np
import pytest
import torch

import oracle
from wavefunctionsimpython_amd import _abi

pytestmark = pytest.mark.gpu

DX, DT = (0.4, 0.35, 0.3), 0.01


def _plan(shape, batch=1):
    return _abi.Plan(shape, DX, DT, 1.0, _abi.WFS_C64, _abi.WFS_METHOD_FOURIER, batch=batch)


def _state(shape, dev, seed):
    rng = np.random.default_rng(seed)
    psi = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    V = rng.uniform(-0.5, 0.5, shape) - 0.05j * rng.random(shape)
    V[..., shape[-3] // 2:, :, :] = V[..., shape[-3] // 2:shape[-3] // 2 + 1, :, :]    # equal x planes
    return torch.from_numpy(psi.astype(np.complex64)).to(dev), torch.from_numpy(V.astype(np.complex64)).to(dev)


# packets of at most 64 planes (4 row groups each) hold at most one group per CU by themselves and more
# together: 72 to 128 planes
@pytest.mark.parametrize("n", [192, 256])
@pytest.mark.parametrize("nx,batch", [(32, 3), (64, 2), (8, 9)])
@pytest.mark.parametrize("separable", [False, True])
@pytest.mark.parametrize("steps", [1, 3])
def test_parts_equal_whole(dev, n, nx, batch, separable, steps):
    shape = (nx, n, n)
    psi, V = _state((batch,) + shape, dev, n + nx)
    axes = [np.random.default_rng(nx).uniform(-1, 1, (batch, m)) for m in shape]
    p = _plan(shape, batch)
    p.set_potential_axes(*axes) if separable else p.set_potential(V)
    a = psi.clone()
    p.step(a, None, steps)
    for i in range(batch):
        q = _plan(shape)
        q.set_potential_axes(*(x[i] for x in axes)) if separable else q.set_potential(V[i].contiguous())
        b = psi[i].clone()
        q.step(b, None, steps)
        assert torch.equal(a[i], b)


@pytest.mark.parametrize("n", [192, 256])
def test_parts_match_oracle(dev, n):
    shape = (96, n, n)
    psi, V = _state(shape, dev, n)
    a = psi.clone()
    _plan(shape).step(a, V, 2)
    ref = oracle.split_step(psi.cpu().numpy(), V.cpu().numpy(), DX, DT, 1.0, nsteps=2)
    # float transforms of length 96, n, n: a few rounding errors of 6e-8 per axis and direction
    assert oracle.relative_l2(a.cpu().numpy(), ref) < 2e-6
