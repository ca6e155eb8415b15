"""I3 tables replaced while a captured graph is alive: the replay takes the new table, also where its terms pair into
mirrors otherwise than those of the table that was captured; a table that is refused leaves the one before it whole."""
import numpy as np
import pytest
import torch

import qbf
from qbf import workloads as wl

pytestmark = pytest.mark.gpu
L, R = wl.L_BOX, wl.R_BALL


def tables(N, J, M, kind):
    """paired: every term has a mirror; some: two pairs broken by weight and one by a phase that is none; single: no
    pairs at all.  Other weights than the paired table's, so that the tables' outputs differ."""
    q = qbf.quadrature(N, J, L, R, M)
    p1, p2 = q[2]
    if kind != "paired":
        p2 *= 1.3
    if kind == "some":
        p2[0] *= 1.5
        p2[1] *= 0.5
        p1[M] *= 1.2
    elif kind == "single":
        p2 *= (1 + 0.1 * np.arange(p2.shape[0]))[:, None, None]
    return q


def step(q, N, prec, pairs, W, h, dt):
    e = qbf.Engine(N, prec, max_cells=W.shape[0])
    e.set_quadrature(*q)
    e.set_real_pairs(pairs, 0.0)
    out = e.inhom_step_periodic(W, L, h, dt)
    torch.cuda.synchronize()
    e.close()
    return out


# the last: five of twelve folded terms a launch (2 GiB of F grids), so that the launches differ too
@pytest.mark.parametrize("N,prec,pairs,n,J,M", [(16, qbf.FP64, 0, 3, 4, 4), (32, qbf.FP32, 0, 2, 4, 3), (64, qbf.FP32, 2, 3, 4, 2),
                                                (64, qbf.FP64, 2, 1, 4, 2), (128, qbf.FP32, 0, 2, 4, 2), (16, qbf.FP64, 0, 6500, 4, 6)])
@pytest.mark.parametrize("first,then", [("paired", "some"), ("paired", "single"), ("single", "paired"), ("some", "paired")])
def test_replay_takes_the_new_table(N, prec, pairs, n, J, M, first, then):
    print(f"N = {N}, precision {prec}, pairs {pairs}, {n} cells, {first} -> {then}", flush=True)
    h, dt = 1.0 / n, 1e-3 / n
    W = torch.from_numpy(wl.periodic(N, min(n, 8), seed=2)).cuda()
    W = W.repeat((n + 7) // 8, 1, 1, 1)[:n].contiguous()
    a, b = tables(N, J, M, first), tables(N, J, M, then)
    refs = [step(q, N, prec, pairs, W, h, dt) for q in (a, b)]
    apart = (refs[0] - refs[1]).norm()
    # the same step with the terms in another order: rounding (of the convolutions: FP32, or FP64) against what
    # the tables' difference makes
    tol = 1e-9 if prec == qbf.FP64 else 1e-3
    e = qbf.Engine(N, prec, max_cells=n)
    e.set_quadrature(*a)
    e.set_real_pairs(pairs, 0.0)
    Win = W.clone()
    g, out = e.capture_inhom_step_periodic(Win, L, h, dt)
    for q, ref in ((b, refs[1]), (a, refs[0]), (b, refs[1])):
        e.set_quadrature(*q)
        for _ in range(2):
            out.zero_()
            Win.copy_(W)
            torch.cuda.synchronize()
            g.launch()
            torch.cuda.synchronize()
            assert (out - ref).norm() < tol * apart
        # eager, in the buffers that the graph pins
        assert (e.inhom_step_periodic(W, L, h, dt) - ref).norm() < tol * apart
    # more terms than the buffers hold: refused, and nothing is written
    with pytest.raises(qbf.QBFError, match="captured graph"):
        e.set_quadrature(*qbf.quadrature(N, J, L, R, M + 2))
    out.zero_()
    g.launch()
    torch.cuda.synchronize()
    assert (out - refs[1]).norm() < tol * apart
    g.close()
    e.close()
