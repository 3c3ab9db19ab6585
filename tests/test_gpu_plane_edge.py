"""Entry and exit transforms of a call as one launch on whole planes against the axis passes: the same bits."""

import numpy as np
import pytest
import torch

from wavefunctionsimpython_amd import _abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [_abi.WFS_C64, _abi.WFS_C128])
@pytest.mark.parametrize("n", [16, 32, 64])
@pytest.mark.parametrize("nx,batch,steps", [(8, 1, 1), (192, 1, 1), (64, 3, 2), (512, 1, 1)])
def test_edges_equal_passes(dev, precision, n, nx, batch, steps):
    rng = np.random.default_rng(n + nx)
    shape = (nx, n, n)
    full = shape if batch == 1 else (batch,) + shape
    dtype = torch.complex128 if precision == _abi.WFS_C128 else torch.complex64
    psi = torch.from_numpy(rng.standard_normal(full) + 1j * rng.standard_normal(full)).to(dev).to(dtype)
    V = torch.from_numpy((rng.uniform(-1, 1, full) - 0.05j * rng.random(full)).astype(np.complex64)).to(dev)
    out = []
    for plane in (1, 0):
        p = _abi.Plan(shape, (0.4, 0.35, 0.3), 0.01, 1.0, precision, _abi.WFS_METHOD_FOURIER, batch=batch)
        p.set_variant("yz_plane", plane)
        p.set_potential(V)
        a = psi.clone()
        p.set_profiling(True)
        p.step(a, None, steps)
        p.step(a, None, 1)             # the next call's table copies
        prof = p.profile(reset=True)
        p.set_profiling(False)
        assert (prof["slab_edge"][0] if "slab_edge" in prof else 0) == (4 if plane else 0)
        out.append(a)
    assert torch.equal(out[0], out[1])
