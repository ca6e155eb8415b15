"""Terms are mirrors when their psi2 agree to rounding on the table's own scale, not on an absolute one."""
import numpy as np
import pytest
import torch

import oracle as O
import qbf
from conftest import l1rel, rand_state

pytestmark = pytest.mark.gpu


def test_small_tables_without_a_value_at_the_origin():
    """psi2 of 1e-14, zero at the origin and beside it, the partners of every pair 1.5 times as large elsewhere."""
    N = 16
    q = O.Quad(N, 4, 6.0, 3.75, 4)
    p1, p2 = q.I3
    p2 = p2.reshape(4, 4, 2 * N, 2 * N)         # a view: the oracle sees it (J, M; m and M - 1 - m are mirrors)
    p2 *= 1e-14
    p2[:, 2:] *= 1.5
    p2[:, :, 0, 0] = p2[:, :, 0, 1] = p2[:, :, 1, 0] = 0
    q.I2[1][:] *= 1e-14
    q.I4[0][:] *= 1e-14
    WF = np.stack([O.r2c_fill(c) for c in rand_state(np.random.default_rng(2), 1, N)[0]])
    ref = O.CdInt(q, WF)
    e = qbf.Engine(N, qbf.FP64, max_cells=1)
    e.set_quadrature(q.I1, q.I2, q.I3, q.I4)
    out = e.collision(torch.from_numpy(WF[None]).cuda(), mode=qbf.CD).cpu().numpy()[0]
    e.close()
    assert l1rel(out, ref) < 1e-12              # rounding, as the other tables; with the pairs taken it is 1e-2 and more
