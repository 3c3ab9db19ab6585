"""complex64 96^2, 128^2 and 512^2 planes stepped as two launches (kernel class yz_split) against the passes, the
slab class's launches and the oracle."""

import numpy as np
import pytest
import torch

import oracle
from wavefunctionsimpython_amd import _abi

pytestmark = pytest.mark.gpu

DX, DT = (0.4, 0.35, 0.3), 0.01
C64 = _abi.WFS_C64


def _plan(shape, split=None, batch=1):
    p = _abi.Plan(shape, DX, DT, 1.0, C64, _abi.WFS_METHOD_FOURIER, batch=batch)
    if split is not None:
        p.set_variant("yz_plane", 0)
        if shape[1] == 128:
            p.set_variant("yz_slab", 0)
        p.set_variant("yz_split", split)
    return p


def _state(shape, dev, seed=0):
    rng = np.random.default_rng(seed)
    psi = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    V = rng.uniform(-0.5, 0.5, shape) - 0.05j * rng.random(shape)
    V[..., shape[-3] // 2:, :, :] = V[..., shape[-3] // 2:shape[-3] // 2 + 1, :, :]    # equal x planes
    return torch.from_numpy(psi.astype(np.complex64)).to(dev), torch.from_numpy(V.astype(np.complex64)).to(dev)


# a few roundings of 6e-8 per transform and axis, steps transforms there and back
@pytest.mark.parametrize("nx,n,steps", [(nx, n, steps) for n in (96, 128)
                                        for nx, steps in ((8, 1), (32, 3), (96, 2), (256, 2))]
                         + [(32, 512, 3), (64, 512, 1), (96, 512, 2), (128, 512, 1), (192, 512, 1), (256, 512, 2),
                            (512, 512, 1)])
def test_split_matches_passes(dev, nx, n, steps):
    shape = (nx, n, n)
    psi, V = _state(shape, dev, n + nx)
    out = []
    for split in (0, 1):
        p = _plan(shape, split)
        a = psi.clone()
        p.step(a, V, steps)            # table of the call
        p.step(a, None, 1)             # table kept
        out.append(a)
    assert oracle.relative_l2(out[1].cpu().numpy(), out[0].cpu().numpy()) < 2e-6


@pytest.mark.parametrize("nx,n", [(16, 96), (16, 128), (32, 512)])
def test_split_matches_oracle_and_follows_the_potential(dev, nx, n):
    shape = (nx, n, n)
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
    assert oracle.relative_l2(a.cpu().numpy(), ref) < 3e-6


# (x launches of few blocks run as lane pairs, a batch's as rows: the same bits at every length of x)
# 3 packets stay below 256 planes of 128^2 (slab class), 10 pass it and the 640 of the 16-z x launch
@pytest.mark.parametrize("shape,batch", [((32, 512, 512), 2), ((16, 96, 96), 3), ((8, 96, 96), 3),
                                         ((32, 96, 96), 3), ((128, 96, 96), 3), ((192, 96, 96), 3), ((256, 96, 96), 3),
                                         ((8, 128, 128), 2), ((96, 128, 128), 2), ((256, 128, 128), 2),
                                         ((64, 96, 96), 10), ((64, 128, 128), 3), ((64, 128, 128), 10)])
def test_default_packets_equal_single_runs(dev, shape, batch):
    rng = np.random.default_rng(batch)
    axes = [rng.uniform(-1, 1, (batch, m)) for m in shape]
    psi = _state((batch,) + shape, dev, batch)[0]
    p = _plan(shape, batch=batch)
    assert p.variants()["yz_split"] or p.variants()["yz_slab"]
    p.set_potential_axes(*axes)
    a = psi.clone()
    p.step(a, None, 3)
    for i in range(batch):
        q = _plan(shape)
        q.set_potential_axes(*(x[i] for x in axes))
        b = psi[i].clone()
        q.step(b, None, 3)
        assert torch.equal(a[i], b)


def test_split_defaults(dev):
    def on(shape, batch=1):
        v = _abi.Plan(shape, DX, DT, 1.0, C64, _abi.WFS_METHOD_FOURIER, batch=batch).variants()
        return v["yz_split"], v["yz_slab"]
    assert on((96, 96, 96)) == (1, 0) and on((8, 96, 96), 40) == (1, 0)
    assert on((128, 128, 128)) == (0, 2) and on((256, 128, 128)) == (1, 0) and on((64, 128, 128), 8) == (1, 0)
    assert on((64, 64, 64)) == (0, 0) and on((512, 64, 64)) == (0, 0) and on((32, 96, 16)) == (0, 0)
    assert on((192, 192, 192)) == (0, 1)
    assert on((512, 512, 512)) == (1, 0) and on((32, 512, 512)) == (1, 0) and on((16, 512, 512)) == (0, 0)
    assert on((512, 256, 256)) == (1, 0) and on((32, 512, 256)) == (1, 0) and on((16, 512, 256)) == (0, 0)
    with pytest.raises(_abi.WfsError):
        _plan((64, 64, 64)).set_variant("yz_split", 1)
