"""Eager calls while a captured graph pins the engine's buffers: fewer cells, single integrals, the other kind of
grids and other tables choose splits that fit the buffers there are; the graph stays valid."""
import numpy as np
import pytest
import torch

import qbf
from conftest import l1rel
from qbf import workloads as wl

pytestmark = pytest.mark.gpu
L, R = wl.L_BOX, wl.R_BALL
TOL = {qbf.FP64: 1e-12, qbf.FP32: 1e-4}       # L1 of the operator: only the order of its sums differs


def engine(N, prec, n, q, pairs=0):
    e = qbf.Engine(N, prec, max_cells=n)
    e.set_quadrature(*q)
    e.set_real_pairs(pairs, 0.0)
    return e


def fourier(N, n):
    W = torch.from_numpy(wl.periodic(N, n, seed=4)).cuda()
    F = torch.fft.fft2(W.to(torch.complex128)) / N ** 2
    F[..., N // 2, :] = 0
    F[..., :, N // 2] = 0
    return W, F.contiguous()


def many_terms(N, J, M):
    """Small I1, I2, I4 tables with J M I3 terms."""
    q = qbf.quadrature(N, 4, L, R, 2)
    p1, p2 = np.empty((J * M, N, N), np.complex128), np.empty((J * M, 2 * N, 2 * N))
    dp = qbf._dp
    qbf.lib().qbf_fourier_I3(N, J, L, R, M, p1.view(np.float64).ctypes.data_as(dp), p2.ctypes.data_as(dp))
    return q[0], q[1], (p1, p2), q[3]


@pytest.mark.parametrize("N,prec,cap,fewer,J,M", [(64, qbf.FP32, 10, (2, 4, 9), 16, 4), (16, qbf.FP64, 33, (16, 32), 16, 4),
                                                  (32, qbf.FP64, 10, (4, 8), 16, 4), (128, qbf.FP32, 10, (4, 8), 8, 8)])
@pytest.mark.parametrize("pairs", [0, 2])
def test_fewer_cells(N, prec, cap, fewer, J, M, pairs):
    print(f"N = {N}, precision {prec}, {cap} cells, pairs {pairs}", flush=True)
    q = qbf.quadrature(N, J, L, R, M)
    W, F = fourier(N, cap)
    refs = {}
    for n in fewer:
        e = engine(N, prec, n, q, pairs)
        refs[n] = e.collision(F[:n].contiguous()).cpu().numpy()
        e.close()
    e = engine(N, prec, cap, q, pairs)
    g, out = e.capture_inhom_step_periodic(W, L, 1 / 64, 1e-4)
    torch.cuda.synchronize()
    first = out.clone()
    for n in fewer:
        assert l1rel(e.collision(F[:n].contiguous()).cpu().numpy(), refs[n]) < TOL[prec], n
    out.zero_()
    g.launch()
    torch.cuda.synchronize()
    assert torch.equal(out, first)
    g.close()
    e.close()


def test_single_integral_and_other_grids():
    """512 terms at N = 64: one cell's step leaves 256 accumulators, the single I3 integral would take 512; 64 cells'
    step on packed pairs fills the F grids, and the complex grids take half as many terms a launch."""
    N = 64
    q = many_terms(N, 32, 16)
    W, F = fourier(N, 64)
    f, h, k = (F[0, c].contiguous() for c in (0, 1, 2))
    e = engine(N, qbf.FP32, 64, q)
    ref3 = e.I3(f, h, k).cpu().numpy()
    refc = e.collision(F).cpu().numpy()
    e.close()
    e = engine(N, qbf.FP32, 1, q)
    e.I2(f, h, k)                         # sizes what the single integrals stage their inputs in
    g, _ = e.capture_inhom_step_periodic(W[:1].contiguous(), L, 1 / 64, 1e-4)
    assert l1rel(e.I3(f, h, k).cpu().numpy(), ref3) < 1e-4
    g.close()
    e.close()
    e = engine(N, qbf.FP32, 64, q, pairs=2)
    g, out = e.capture_inhom_step_periodic(W, L, 1 / 64, 1e-4)
    torch.cuda.synchronize()
    first = out.clone()
    e.set_real_pairs(0, 0.0)
    assert l1rel(e.collision(F).cpu().numpy(), refc) < 1e-4
    out.zero_()
    g.launch()
    torch.cuda.synchronize()
    assert torch.equal(out, first)
    g.close()
    e.close()
