"""A captured plane current, replayed after the plan's workspace grew."""

import pytest
import torch

from wavefunctionsimpython_amd import _abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [_abi.WFS_C64, _abi.WFS_C128])
def test_replay_after_larger_planes(dev, precision):
    shape, dx = (32, 64, 32), (0.4, 0.35, 0.3)
    p = _abi.Plan(shape, dx, 0.01, 1.0, precision, _abi.WFS_METHOD_FOURIER)
    g = torch.Generator(device=dev).manual_seed(2)
    psi = torch.randn(shape, dtype=torch.complex128, device=dev, generator=g)
    psi = psi.to(torch.complex64 if precision == _abi.WFS_C64 else torch.complex128)
    plane = ((0.3, 0.2, -0.1), (1.0, 0.0, 0.0), (8.0, 6.0))
    want = p.plane_current(psi, *plane, (21, 21)).clone()
    out = torch.zeros_like(want)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with _abi.Graph(s) as graph:
        p.plane_current(psi, *plane, (21, 21), out=out, stream=s)
    for count in (21, 101, 501, 31):
        p.plane_current(psi, *plane, (count, count))
        out.zero_()
        torch.cuda.synchronize()
        graph.launch()
        s.synchronize()
        assert torch.equal(out, want), count
        assert torch.equal(p.plane_current(psi, *plane, (21, 21)), want)
