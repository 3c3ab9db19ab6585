"""The network's DFT stages and backward kernels against float64 of the same products.

Bounds, per element, in units of the sum of absolute products: an operand carried as bf16 hi + lo
keeps about 17 bits (2^-17, two operands and the dropped lo lo product: 2^-15.4), FP32 sums of a few
hundred terms in a chain add at most 2^-15: 2^-14 covers both.
"""

import numpy as np
import pytest
import torch

from wavefunctionsimpython_amd import _abi
from wavefunctionsimpython_amd.fno import dft_tables

pytestmark = pytest.mark.gpu

BOUND = 2.0 ** -14


def _bf16(x):
    return torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(torch.bfloat16).double().numpy()


def _dev(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x, np.float32)).to(dev)


@pytest.mark.parametrize("C,cin,P", [(32, 32, 32768), (32, 32, 32), (2, 32, 4096), (32, 5, 110592), (1, 1, 96),
                                     (17, 20, 992)])
def test_weight_grad(dev, C, cin, P):
    rng = np.random.default_rng(C + P)
    g, v = rng.standard_normal((C, P)), rng.standard_normal((cin, P))
    gW, gb = rng.standard_normal((C, cin)), rng.standard_normal(C)
    t = [_dev(x, dev) for x in (g, v, gW, gb)]
    work = torch.empty(_abi.WEIGHT_GRAD_WORK, dtype=torch.float32, device=dev)
    _abi.fno_weight_grad(*t, C, cin, P, work)
    g, v, gW, gb = (np.float64(np.float32(x)) for x in (g, v, gW, gb))
    eW = np.abs(t[2].cpu().numpy() - (gW + g @ v.T)) / (np.abs(gW) + np.abs(g) @ np.abs(v).T)
    eb = np.abs(t[3].cpu().numpy() - (gb + g.sum(1))) / (np.abs(gb) + np.abs(g).sum(1))
    assert eW.max() < BOUND and eb.max() < BOUND


def test_weight_grad_limits(dev):
    z = torch.zeros(33 * 64, device=dev)
    work = torch.empty(_abi.WEIGHT_GRAD_WORK, dtype=torch.float32, device=dev)
    for C, P, w in ((33, 64, work), (2, 48, work), (2, 64, work[:100])):
        with pytest.raises(_abi.WfsError):
            _abi.fno_weight_grad(z, z, z, z, C, 1, P, w)


@pytest.mark.parametrize("C,m3", [(32, 1728), (5, 8), (40, 27), (1, 1)])
def test_modes_backward(dev, C, m3):
    rng = np.random.default_rng(C)
    Rr, Ri, gr, gi = (rng.standard_normal((m3, C, C)) for _ in range(4))
    X, dO = (rng.standard_normal((C, 2, m3)) for _ in range(2))
    t = [_dev(x, dev) for x in (Rr, Ri, X, dO, np.zeros_like(X), gr, gi)]
    _abi.fno_modes_backward(*t, m3, C)
    Rr, Ri = _bf16(Rr), _bf16(Ri)
    X, dO, gr, gi = (x.astype(np.float32).astype(np.float64) for x in (X, dO, gr, gi))
    (xr, xi), (dr, di) = X.transpose(1, 2, 0), dO.transpose(1, 2, 0)          # [q][c]
    want = {5: gr + xr[:, :, None] * dr[:, None] + xi[:, :, None] * di[:, None],
            6: gi + xr[:, :, None] * di[:, None] - xi[:, :, None] * dr[:, None]}
    for k, ref in want.items():
        assert np.abs(t[k].cpu().numpy() - ref).max() < BOUND * np.abs(ref).max()
    dX = np.stack([(Rr * dr[:, None] + Ri * di[:, None]).sum(2), (Rr * di[:, None] - Ri * dr[:, None]).sum(2)])
    scale = (np.abs(Rr) * np.abs(dr[:, None]) + np.abs(Ri) * np.abs(di[:, None])).sum(2).max()
    assert np.abs(t[4].cpu().numpy().transpose(1, 2, 0) - dX).max() < BOUND * scale


# reducing (M <= 32) and expanding (K <= 32) stages, few and many columns, partial tiles of both
@pytest.mark.parametrize("M,K,ncol,slabs", [(24, 256, 12, 96), (24, 128, 144, 5), (256, 24, 144, 5), (128, 32, 16, 2000),
                                           (12, 96, 6, 7), (96, 12, 6, 7), (32, 16, 1, 1), (16, 8, 3, 50),
                                           (64, 4, 4, 1)])
def test_dft_stage(dev, M, K, ncol, slabs):
    rng = np.random.default_rng(M + K)
    A = rng.uniform(-1, 1, (M, K))
    src = rng.standard_normal((slabs, K, ncol))
    dst = torch.full((slabs * M * ncol + 64,), 7.0, dtype=torch.float32, device=dev)
    _abi.fno_stage(_abi.fno_stage_table(A, dev), _dev(src, dev), dst, M, K, ncol, slabs)
    x = np.float64(np.float32(src))
    got = dst.double().cpu().numpy()
    ref, scale = np.matmul(_bf16(A), x), np.matmul(np.abs(_bf16(A)), np.abs(x))
    assert (np.abs(got[:-64].reshape(slabs, M, ncol) - ref) <= BOUND * scale).all()
    assert (got[-64:] == 7.0).all()


@pytest.mark.parametrize("n,C,cin,m,spectral,factor", [(32, 32, 32, 12, True, True), (64, 20, 20, 6, True, True),
                                                       (96, 7, 2, 16, False, False), (128, 4, 4, 10, True, False)])
def test_layer_backward(dev, n, C, cin, m, spectral, factor):
    rng = np.random.default_rng(n)
    tm, P = 2 * m, n ** 3
    tab = dft_tables(n, m)
    W, g = rng.standard_normal((cin, C)), rng.standard_normal((cin, P))
    Tg, u = rng.standard_normal((C, n * n, tm)), rng.standard_normal((C, P))
    W_, g_, Tg_, u_, Gz, Fz = (_dev(x, dev) for x in (W, g, Tg, u, tab["Gz"], tab["Fz"]))
    gn = torch.empty(C * P, dtype=torch.float32, device=dev)
    Tn = torch.empty(C * n * n * tm, dtype=torch.float32, device=dev)
    _abi.fno_layer_backward(W_, g_, Tg_ if spectral else None, u_ if factor else None, Gz, Fz, gn, Tn, cin, C, n, tm)
    Wd, gd, Td, Fd, Gd = (torch.from_numpy(x).to(dev) for x in
                          (_bf16(W), np.float64(np.float32(g)), np.float64(np.float32(Tg)), _bf16(tab["Fz"]),
                           _bf16(tab["Gz"])))
    ref, scale = Wd.t() @ gd, Wd.abs().t() @ gd.abs()
    if spectral:
        ref = ref + (Td.reshape(-1, tm) @ Fd.t()).reshape(C, P)
        scale = scale + (Td.abs().reshape(-1, tm) @ Fd.abs().t()).reshape(C, P)
    if factor:
        x = u_.double().requires_grad_(True)
        (f,) = torch.autograd.grad(torch.nn.functional.gelu(x, approximate="tanh").sum(), x)
        ref, scale = ref * f, scale * f.abs().clamp_min(0.1)      # the hardware exponential errs a few ulp of 1
    got = gn.double().reshape(C, P)
    assert float(((got - ref).abs() / scale).max()) < BOUND
    want = got.reshape(-1, n) @ Gd.t()
    tscale = got.abs().reshape(-1, n) @ Gd.abs().t()
    # (the sine of frequency 0 is zero on both sides)
    assert bool(((Tn.double().reshape(-1, tm) - want).abs() <= BOUND * tscale).all())


@pytest.mark.parametrize("n,C,cin,cout,m,spectral,residual,keep", [(32, 32, 32, 2, 12, True, True, False),
                                                                   (64, 20, 20, 1, 6, True, False, True),
                                                                   (96, 7, 5, 2, 16, False, True, True)])
def test_last_layer(dev, n, C, cin, cout, m, spectral, residual, keep):
    rng = np.random.default_rng(n + cout)
    tm, P = 2 * m, n ** 3
    Gz = dft_tables(n, m)["Gz"]
    W, v, b = rng.standard_normal((C, cin)), rng.standard_normal((cin, P)), rng.standard_normal(C)
    Z, Q, qb = rng.standard_normal((C, n * n, tm)), rng.standard_normal((cout, C)), rng.standard_normal(cout)
    base = rng.standard_normal((cout, P))
    W_, v_, b_, Z_, Gz_, Q_, qb_, base_ = (_dev(x, dev) for x in (W, v, b, Z, Gz, Q, qb, base))
    u = torch.empty(C * P, dtype=torch.float32, device=dev) if keep else None
    out = torch.empty(cout * P, dtype=torch.float32, device=dev)
    _abi.fno_last_layer(W_, v_, Z_ if spectral else None, b_, Gz_, Q_, qb_, base_ if residual else None, 0.5, u, out,
                        cin, C, cout, n, tm)
    Wd, Gd, Qd = (torch.from_numpy(_bf16(x)).to(dev) for x in (W, Gz, Q))
    ref = Wd @ v_.double() + b_.double()[:, None]
    scale = Wd.abs() @ v_.double().abs() + b_.double().abs()[:, None]
    if spectral:
        ref = ref + (Z_.double().reshape(-1, tm) @ Gd).reshape(C, P)
        scale = scale + (Z_.double().abs().reshape(-1, tm) @ Gd.abs()).reshape(C, P)
    if keep:
        assert bool(((u.double().reshape(C, P) - ref).abs() <= BOUND * scale).all())
    want = 0.5 * (Qd @ ref + qb_.double()[:, None]) + (base_.double() if residual else 0.0)
    oscale = Qd.abs() @ scale + qb_.double().abs()[:, None] + base_.double().abs()
    assert bool(((out.double().reshape(cout, P) - want).abs() <= BOUND * oscale).all())
