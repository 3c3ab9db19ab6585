"""The autotuner on grids that may step in two launches (kernel class yz_split)."""

import pytest
import torch

from wavefunctionsimpython_amd import _abi

pytestmark = pytest.mark.gpu

DX, DT = (0.4, 0.35, 0.3), 0.01


# grids on which the two launches take at most 0.7 of the passes' time, so that the choice is not one of noise
@pytest.mark.parametrize("shape,precision", [((64, 192, 192), _abi.WFS_C128), ((96, 192, 128), _abi.WFS_C64),
                                             ((64, 96, 96), _abi.WFS_C64)])
def test_autotune_compares_the_two_launches(dev, shape, precision):
    p = _abi.Plan(shape, DX, DT, 1.0, precision, _abi.WFS_METHOD_FOURIER)
    assert p.variants()["yz_split"] == 1
    p.set_variant("yz_split", 0)
    assert p.autotune()["yz_split"] == 1
    g = torch.Generator(device=dev).manual_seed(3)
    V = (torch.rand(shape, device=dev, generator=g) - 0.5).to(torch.complex64)
    psi = torch.randn(shape, dtype=torch.complex128, device=dev, generator=g)
    psi = psi.to(torch.complex128 if precision == _abi.WFS_C128 else torch.complex64)
    want = psi.clone()
    p.step(psi, V, 3)
    _abi.Plan(shape, DX, DT, 1.0, precision, _abi.WFS_METHOD_FOURIER).step(want, V, 3)
    assert torch.equal(psi, want)
