"""CdInt with its I3 terms taken in mirrored pairs (one pass per pair) against the oracle's term-by-term
sum, over the tables the pairing accepts and refuses, and over the kernels' splits of the terms."""
import numpy as np
import pytest
import torch

import oracle as O
import qbf
from conftest import l1rel, rand_state

pytestmark = pytest.mark.gpu
L, R = 6.0, 3.75
TOL64, TOL32 = 1e-12, 1e-4      # L1 of Cd: rounding; the FP32 convolution path


def tables(kind, N, J, M):
    """The reference's tables, with the I3 terms' order or pairing changed (in place: the oracle sees them)."""
    q = O.Quad(N, J, L, R, M)
    p1, p2 = q.I3
    n = p2.shape[0]
    rng = np.random.default_rng(7)
    if kind == "permuted":
        o = rng.permutation(n)
        p1[:], p2[:] = p1[o], p2[o]
    elif kind == "unpaired":              # every second term of a pair with another weight: no mirrors
        p2 *= (1 + 0.1 * np.arange(n))[:, None, None].reshape((n,) + (1,) * (p2.ndim - 1))
    elif kind == "some":                  # a part of the pairs broken: by weight, and by a phase that is none
        p2[0] *= 1.5
        p1[1] *= 1.1
    return q


def engine(q, N, prec, n, pairs=None):
    e = qbf.Engine(N, prec, max_cells=n)
    e.set_quadrature(q.I1, q.I2, q.I3, q.I4)
    if pairs is not None:
        e.set_real_pairs(pairs, 2e-5)
    return e


def fourier(W):
    return np.stack([[O.r2c_fill(c) for c in w] for w in W])


@pytest.mark.parametrize("N,J,M,n", [(16, 4, 2, 1), (16, 4, 5, 3), (32, 6, 4, 2), (64, 4, 3, 1)])
@pytest.mark.parametrize("kind", ["plain", "permuted", "unpaired", "some"])
def test_cd_vs_oracle(kind, N, J, M, n):
    q = tables(kind, N, J, M)
    WF = fourier(rand_state(np.random.default_rng(N + n), n, N))
    ref = np.stack([O.CdInt(q, w) for w in WF])
    W = torch.from_numpy(WF).cuda()
    for prec, pairs, tol in ((qbf.FP64, 0, TOL64), (qbf.FP32, 0, TOL32)):
        e = engine(q, N, prec, n, pairs)
        out = e.collision(W, mode=qbf.CD).cpu().numpy()
        e.close()
        assert l1rel(out, ref) < tol, (kind, prec)


@pytest.mark.parametrize("N,J,M", [(16, 4, 3), (32, 4, 4), (64, 4, 2)])
def test_packed_pairs_on_nyquist_free_spectra(N, J, M):
    """The packed pairs' mirror sums (and their +N/2 edge) against the oracle, both precisions."""
    q = tables("plain", N, J, M)
    WF = fourier(rand_state(np.random.default_rng(3), 2, N))
    WF[..., N // 2, :] = 0
    WF[..., :, N // 2] = 0
    ref = np.stack([O.CdInt(q, w) for w in WF])
    W = torch.from_numpy(WF).cuda()
    for prec, tol in ((qbf.FP64, TOL64), (qbf.FP32, TOL32)):
        e = engine(q, N, prec, 2, 2)
        out = e.collision(W, mode=qbf.CD).cpu().numpy()
        e.close()
        assert l1rel(out, ref) < tol


def test_several_launches_accumulate():
    """96 cells need two launches of the I3 terms (F grids of 2 GiB each); the same cells one by one
    need one, with the terms split over workgroups: only the order of the sums differs."""
    N, n = 32, 96
    q = qbf.quadrature(N, 16, L, R, 16)
    W = torch.fft.fft2(torch.from_numpy(rand_state(np.random.default_rng(5), n, N)).cuda().to(torch.complex128)) / N ** 2
    e = qbf.Engine(N, qbf.FP64, max_cells=n)
    e.set_quadrature(*q)
    out = e.collision(W, mode=qbf.CD)
    assert torch.equal(out, e.collision(W, mode=qbf.CD))
    for c in (0, 47, 95):
        one = e.collision(W[c:c + 1].contiguous(), mode=qbf.CD)
        assert l1rel(one.cpu().numpy()[0], out[c].cpu().numpy()) < TOL64
    e.close()
