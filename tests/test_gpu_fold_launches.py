"""The mirrored I3 terms over several launches: blocks of mirror sums that a launch holds (many terms per launch) or
that several launches fill together (many cells, few terms per launch), the last launch shorter, both kinds of
grids; and the device memory they take."""
import numpy as np
import pytest
import torch

import oracle as O
import qbf
from conftest import l1rel, rand_state

pytestmark = pytest.mark.gpu
L, R = 6.0, 3.75
TOL32 = 1e-4      # L1 of Cd, the FP32 convolution path; a block missing or taken twice is 1e-2 or more


def few_then_many(N, n, distinct=4, seed=3):
    """n Fourier states, `distinct` ones repeated, with empty Nyquist lines (either kind of grids is exact)."""
    W = rand_state(np.random.default_rng(seed), distinct, N)
    W = torch.fft.fft2(torch.from_numpy(W).cuda().to(torch.complex128)) / N ** 2
    W[..., N // 2, :] = 0
    W[..., :, N // 2] = 0
    return W.repeat((n + distinct - 1) // distinct, 1, 1, 1)[:n].contiguous()


def reference(q, W, N):
    e = qbf.Engine(N, qbf.FP64, max_cells=W.shape[0])
    e.set_quadrature(*q)
    out = e.collision(W.contiguous(), mode=qbf.CD)
    e.close()
    return out


# F grids of 8 GiB a launch.  Complex grids: N = 64, 700 cells: 24 of 64 terms, then 24 and 16; 4096 cells: 4 of 18;
# N = 32, 2500 cells: 27 terms; N = 128, 700 cells: 2 terms.  Packed pairs: twice as many.
@pytest.mark.parametrize("pairs", [0, 2])
@pytest.mark.parametrize("N,n,J,M", [(64, 700, 8, 16), (64, 4096, 6, 6), (32, 2500, 8, 16), (128, 700, 4, 14)])
def test_launches_and_blocks(N, n, J, M, pairs):
    print(f"N = {N}, {n} cells, pairs {pairs}", flush=True)
    q = qbf.quadrature(N, J, L, R, M)
    W = few_then_many(N, n)
    ref = reference(q, W[:4], N).cpu().numpy()
    e = qbf.Engine(N, qbf.FP32, max_cells=n)
    e.set_quadrature(*q)
    e.set_real_pairs(pairs, 0.0)
    out = e.collision(W, mode=qbf.CD)
    for c in (0, 1, n // 2, n - 2, n - 1):
        assert l1rel(out[c].cpu().numpy(), ref[c % 4]) < TOL32, c
    assert torch.equal(out, e.collision(W, mode=qbf.CD))
    e.close()


def test_memory_does_not_grow_with_the_terms():
    """1024 cells, 32 and 128 folded terms: the same launches' worth of F grids and mirror sums."""
    N, n = 64, 1024
    W = few_then_many(N, n)
    used = []
    for M in (4, 16):
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        e = qbf.Engine(N, qbf.FP32, max_cells=n)
        e.set_quadrature(*qbf.quadrature(N, 16, L, R, M))
        e.set_real_pairs(0, 0.0)
        out = torch.empty_like(W)
        e.collision(W, mode=qbf.CD, out=out)
        torch.cuda.synchronize()
        used.append(free - torch.cuda.mem_get_info()[0])
        e.close()
        del out
        torch.cuda.empty_cache()
    print("GiB:", [u / 2 ** 30 for u in used], flush=True)
    assert used[1] - used[0] < 2 ** 30           # (the tables: 50 MB)


# a part of the pairs broken at N = 128: terms without a mirror between mirrored ones
@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-4)])
def test_unpaired_terms_at_n128(prec, tol):
    N = 128
    q = O.Quad(N, 2, L, R, 6)
    q.I3[1][0] *= 1.5
    q.I3[0][7] *= 1.1
    WF = np.stack([[O.r2c_fill(c) for c in w] for w in rand_state(np.random.default_rng(1), 1, N)])
    ref = O.CdInt(q, WF[0])
    e = qbf.Engine(N, {"fp64": qbf.FP64, "fp32": qbf.FP32}[prec], max_cells=1)
    e.set_quadrature(q.I1, q.I2, q.I3, q.I4)
    e.set_real_pairs(0, 0.0)
    assert l1rel(e.collision(torch.from_numpy(WF).cuda(), mode=qbf.CD).cpu().numpy()[0], ref) < tol
    e.close()


def test_memory_of_a_step():
    """1024 cells at N = 64, FP32, complex grids, 4 folded terms: 2 GiB of F grids, 19 padded grids a cell (2.4 GiB), the
    states (1.0), the mirror sums (0.75), 0.1 of tables and code, in all 6.3; the sums that k_combine transforms have
    no grids of their own (0.5 more)."""
    from qbf import workloads as wl
    N, n = 64, 1024
    W = torch.from_numpy(wl.periodic(N, 64, seed=1)).cuda().repeat(16, 1, 1, 1)
    q = qbf.quadrature(N, 4, L, R, 2)
    out = torch.empty_like(W)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    e = qbf.Engine(N, qbf.FP32, max_cells=n)
    e.set_quadrature(*q)
    e.set_real_pairs(0, 0.0)
    e.inhom_step_periodic(W, L, 1 / n, wl.cfl_dt(N, n), out=out)
    torch.cuda.synchronize()
    used = (free - torch.cuda.mem_get_info()[0]) / 2 ** 30
    e.close()
    print(f"{used:.2f} GiB", flush=True)
    assert used < 6.55
