"""The line transforms over 4, 8 and 16 lanes: state transforms against numpy on rough data, the grids of
the collision operator against the oracle, and the term ranges of many-cell evaluations."""
import numpy as np
import pytest
import torch

import oracle as O
import qbf
from conftest import l1rel, rand_state

pytestmark = pytest.mark.gpu
L, R = 6.0, 3.75


@pytest.mark.parametrize("N", [16, 32, 64, 128])
def test_state_transforms(N):
    # rounding of 2 log2 N radix-2 stages: a few eps in L1; 1e-14 leaves a factor of ten
    W = np.random.default_rng(N).standard_normal((3, 4, N, N))
    e = qbf.Engine(N, qbf.FP64, max_cells=3)
    F = e.phys_to_fourier(torch.from_numpy(W).cuda())
    assert l1rel(F.cpu().numpy(), np.fft.fft2(W) / N ** 2) < 1e-14
    assert l1rel(e.fourier_to_phys(F).cpu().numpy(), W) < 1e-14
    e.close()


# FP32: rounding of float, 1e-4 of Cc + Cd as the other FP32 parity tests
@pytest.mark.parametrize("N,J,M", [(16, 4, 3), (32, 4, 3), (64, 4, 2)])
@pytest.mark.parametrize("prec,pairs,tol", [("fp64", 0, 1e-12), ("fp64", 2, 1e-12), ("fp32", 0, 1e-4), ("fp32", 2, 1e-4), ("bf16x3", 0, 1e-4)])
def test_collision_vs_oracle(N, J, M, prec, pairs, tol):
    if prec == "bf16x3" and N != 64:
        pytest.skip("N = 64 only")
    q = O.Quad(N, J, L, R, M)
    WF = np.stack([[O.r2c_fill(c) for c in w] for w in rand_state(np.random.default_rng(N), 3, N)])
    if pairs:                                  # the packed path drops the Nyquist lines' imaginary parts
        WF[..., N // 2, :] = 0
        WF[..., :, N // 2] = 0
    ref = np.stack([O.CdInt(q, w) for w in WF])
    e = qbf.Engine(N, {"fp64": qbf.FP64, "fp32": qbf.FP32, "bf16x3": qbf.BF16X3}[prec], max_cells=3)
    e.set_quadrature(q.I1, q.I2, q.I3, q.I4)
    e.set_real_pairs(pairs, 2e-5)
    assert l1rel(e.collision(torch.from_numpy(WF).cuda(), mode=qbf.CD).cpu().numpy(), ref) < tol
    e.close()


@pytest.mark.parametrize("N,n,J,M", [(16, 520, 8, 4), (32, 131, 4, 8), (32, 64, 4, 8)])
def test_many_cells(N, n, J, M):
    """Several term ranges per cell on a full chip: only the order of the sums differs from one cell's."""
    W = torch.fft.fft2(torch.from_numpy(rand_state(np.random.default_rng(5), n, N)).cuda().to(torch.complex128)) / N ** 2
    e = qbf.Engine(N, qbf.FP64, max_cells=n)
    e.set_quadrature(*qbf.quadrature(N, J, L, R, M))
    out = e.collision(W, mode=qbf.CD)
    for c in (0, n // 2, n - 1):
        one = e.collision(W[c:c + 1].contiguous(), mode=qbf.CD)
        assert l1rel(one.cpu().numpy()[0], out[c].cpu().numpy()) < 1e-12
    e.close()
