"""The per-axis tables of a separable potential: refused and repeated settings."""

import numpy as np
import pytest
import torch

from wavefunctionsimpython_amd import _abi

pytestmark = pytest.mark.gpu

DX, DT = (0.4, 0.35, 0.3), 0.01
C64, C128 = _abi.WFS_C64, _abi.WFS_C128
# axis passes, plane pass, slab scheme, planes of unequal sides, complex128 planes
GRIDS = [((32, 16, 64), C64), ((32, 64, 64), C64), ((16, 128, 128), C64), ((32, 64, 96), C64), ((16, 64, 64), C128)]


def _axes(shape, seed):
    rng = np.random.default_rng(seed)
    return [rng.uniform(-1, 1, m) for m in shape]


def _plan(shape, precision):
    return _abi.Plan(shape, DX, DT, 1.0, precision, _abi.WFS_METHOD_FOURIER)


def _state(shape, precision, dev):
    g = torch.Generator(device=dev).manual_seed(1)
    psi = torch.randn(shape, dtype=torch.complex128, device=dev, generator=g)
    return psi.to(torch.complex64 if precision == C64 else torch.complex128)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("shape,precision", GRIDS)
def test_refused_axes_leave_the_potential(dev, shape, precision, axis):
    first, second = _axes(shape, 1), _axes(shape, 2)
    second[axis][shape[axis] // 2] = np.inf
    start = _state(shape, precision, dev)
    out = []
    for refused in (False, True):
        p = _plan(shape, precision)
        p.set_potential_axes(*first)
        if refused:
            with pytest.raises(_abi.WfsError):
                p.set_potential_axes(*second)
        out.append(start.clone())
        p.step(out[-1], None, 2)
    torch.cuda.synchronize()
    assert torch.equal(*out)


@pytest.mark.parametrize("shape,precision", GRIDS)
def test_replay_reads_axes_set_after_its_capture(dev, shape, precision):
    start = _state(shape, precision, dev)
    p = _plan(shape, precision)
    p.set_potential_axes(*_axes(shape, 1))
    psi = start.clone()
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with _abi.Graph(s) as graph:
        p.step(psi, None, 2, stream=s)
    for seed in (1, 2, 3, 1):
        axes = _axes(shape, seed)
        p.set_potential_axes(*axes)
        psi.copy_(start)
        torch.cuda.synchronize()
        graph.launch()
        s.synchronize()
        q = _plan(shape, precision)                    # the table copies of a first call, as in the capture
        q.set_potential_axes(*axes)
        want = start.clone()
        q.step(want, None, 2)
        torch.cuda.synchronize()
        assert torch.equal(psi, want), seed
