"""Power series: fused stages on every window form against one launch per stage (same bits)."""

import numpy as np
import pytest
import torch

from wavefunctionsimpython_amd import _abi

pytestmark = pytest.mark.gpu

C64, C128 = _abi.WFS_C64, _abi.WFS_C128


# window forms (whole rows, tiles of 64 and 128 columns, small blocks), partial last tiles, x slabs of
# one plane, faces inside a strip of rows, orders that end in 1, 2 and 3 stages, one to three steps
@pytest.mark.parametrize("precision,n,order,batch,nsteps", [
    (C64, (8, 16, 256), 10, 1, 2), (C64, (8, 32, 192), 9, 1, 1), (C64, (16, 8, 512), 8, 1, 3),
    (C64, (32, 192, 128), 7, 1, 2), (C64, (64, 96, 96), 3, 1, 1), (C64, (64, 64, 64), 5, 1, 2),
    (C64, (16, 16, 64), 1, 3, 2), (C64, (512, 8, 8), 2, 1, 1), (C64, (8, 512, 16), 6, 1, 2),
    (C128, (8, 64, 256), 10, 1, 2), (C128, (16, 16, 512), 7, 1, 1), (C128, (64, 96, 128), 7, 1, 3),
    (C128, (32, 8, 64), 4, 2, 1), (C128, (8, 8, 8), 1, 1, 2)])
def test_fused_stages_equal_single_stages(dev, precision, n, order, batch, nsteps):
    shape = tuple(n) if batch == 1 else (batch,) + tuple(n)
    rng = np.random.default_rng(7)
    psi = torch.from_numpy((rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) * 0.1)
    psi = psi.to(dev, torch.complex128 if precision == C128 else torch.complex64).contiguous()
    V = torch.from_numpy((rng.uniform(-0.5, 0.5, shape) - 0.05j * rng.random(shape)).astype(np.complex64)).to(dev)
    states = []
    for variant in (0, 1, 2):
        plan = _abi.Plan(n, (0.4, 0.4, 0.4), 0.01, 1.0, precision, _abi.WFS_METHOD_POWER_SERIES, order=order,
                         batch=batch)
        plan.set_variant("horner_stage", variant)
        states.append(psi.clone())
        plan.step(states[-1], V, nsteps)
    torch.cuda.synchronize()
    assert torch.equal(states[0], states[1]) and torch.equal(states[0], states[2])
