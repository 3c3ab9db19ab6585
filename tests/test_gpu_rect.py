"""complex64 planes of unequal sides, and square planes beside 512 x planes, stepped as two launches against
the axis passes and the oracle."""

import numpy as np
import pytest
import torch

import oracle
from wavefunctionsimpython_amd import _abi

pytestmark = pytest.mark.gpu

DX, DT = (0.4, 0.35, 0.3), 0.01
C64 = _abi.WFS_C64
SIDES = (32, 64, 96, 128, 192, 256, 512)
PLANES = [(ny, nz) for ny in SIDES for nz in SIDES if ny != nz]
# a few roundings of 6e-8 per transform and axis, steps transforms there and back
TOL = 2e-6


def _plan(shape, split=None, batch=1):
    p = _abi.Plan(shape, DX, DT, 1.0, C64, _abi.WFS_METHOD_FOURIER, batch=batch)
    if split is not None:
        p.set_variant("yz_split", split)
    return p


def _state(shape, dev, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed)
    psi = torch.randn(shape, dtype=torch.complex64, device=dev, generator=g)
    V = torch.rand(shape, device=dev, generator=g) - 0.5 - 0.05j * torch.rand(shape, device=dev, generator=g)
    V[..., shape[-3] // 2:, :, :] = V[..., shape[-3] // 2:shape[-3] // 2 + 1, :, :]    # equal x planes
    return psi, V


def _compare(shape, dev, separable):
    psi, V = _state(shape, dev, sum(shape))
    axes = [np.random.default_rng(a).uniform(-1, 1, (1, m)) for a, m in enumerate(shape)]
    out = []
    for split in (0, 1):
        p = _plan(shape, split)
        p.set_potential_axes(*axes) if separable else p.set_potential(V)
        a = psi.clone()
        p.step(a, None, 2)
        p.step(a, None, 1)
        out.append(a)
    return float((out[1] - out[0]).norm() / out[0].norm())


@pytest.mark.parametrize("separable", [False, True])
@pytest.mark.parametrize("ny,nz", PLANES)
def test_planes_match_passes(dev, ny, nz, separable):
    assert _compare((32, ny, nz), dev, separable) < TOL


# one plane of each number of residue classes (1, 2, 4, 8) beside every length of x
@pytest.mark.parametrize("nx", [8, 16, 32, 64, 96, 128, 192, 256, 512])
@pytest.mark.parametrize("ny,nz", [(32, 128), (64, 96), (256, 96), (512, 64), (96, 512)])
def test_x_lengths_match_passes(dev, nx, ny, nz):
    if _plan((nx, ny, nz)).variants()["yz_split"] == 0:
        assert nx < 32 and (ny, nz) == (96, 512)      # 8 rows need 8 points of an x line in a lane
        return
    assert _compare((nx, ny, nz), dev, False) < TOL


@pytest.mark.parametrize("n", [96, 128, 192, 256])
def test_long_x_matches_passes(dev, n):
    assert _compare((512, n, n), dev, False) < TOL


@pytest.mark.parametrize("shape", [(16, 96, 128), (8, 256, 32), (32, 64, 512)])
def test_matches_oracle_and_follows_the_potential(dev, shape):
    psi, V = _state(shape, dev, 3)
    p = _plan(shape, 1)
    a = psi.clone()
    p.set_potential(V)
    p.step(a, None, 2)
    W = V.clone()
    W[3:5] *= 0.5
    p.set_potential_planes(W, 3, 5)
    p.step(a, None, 2)
    p.set_variant("yz_split", 0)       # the table moves to the passes' order and back
    p.step(a, None, 1)
    p.set_variant("yz_split", 1)
    p.step(a, None, 1)
    ref = oracle.split_step(psi.cpu().numpy(), V.cpu().numpy(), DX, DT, 1.0, nsteps=2)
    ref = oracle.split_step(ref, W.cpu().numpy(), DX, DT, 1.0, nsteps=4)
    assert oracle.relative_l2(a.cpu().numpy(), ref) < 2 * TOL


@pytest.mark.parametrize("shape,batch", [((8, 32, 64), 5), ((16, 96, 128), 3), ((32, 192, 64), 2)])
def test_packets_equal_single_runs(dev, shape, batch):
    rng = np.random.default_rng(batch)
    axes = [rng.uniform(-1, 1, (batch, m)) for m in shape]
    psi = _state((batch,) + shape, dev, batch)[0]
    p = _plan(shape, batch=batch)
    assert p.variants()["yz_split"] == 1
    p.set_potential_axes(*axes)
    a = psi.clone()
    p.step(a, None, 3)
    for i in range(batch):
        q = _plan(shape)
        q.set_potential_axes(*(x[i] for x in axes))
        b = psi[i].clone()
        q.step(b, None, 3)
        assert torch.equal(a[i], b)
