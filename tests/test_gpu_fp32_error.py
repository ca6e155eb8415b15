"""The error of FP32 collision steps against 64 bits.  The bounds are the errors that the same steps had with every I3
term transformed and summed by itself in FP32: taking the terms in mirrored pairs must not cost accuracy."""
import numpy as np
import pytest
import torch

import qbf
from conftest import l1rel
from qbf import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,n,J,M,Nx,pairs,kmax,bound", [
    (64, 10, 32, 16, 512, None, 4, 1.399e-9), (64, 10, 32, 16, 512, 0, 4, 1.218e-9), (64, 300, 12, 6, 512, None, 4, 1.256e-9),
    (32, 64, 32, 16, 512, None, 4, 6.94e-10), (32, 64, 32, 16, 512, 0, 4, 5.85e-10), (128, 8, 16, 8, 2048, 0, 8, 5.94e-10)])
def test_fp32_step_error(N, n, J, M, Nx, pairs, kmax, bound):
    q = qbf.quadrature(N, J, wl.L_BOX, wl.R_BALL, M)
    dt = wl.cfl_dt(64, Nx)
    err = []
    for seed in (100, 101):
        W = torch.from_numpy(wl.periodic(N, n, seed=seed, kmax=kmax)).cuda()
        out = []
        for prec in (qbf.FP64, qbf.FP32):
            e = qbf.Engine(N, prec, max_cells=n)
            e.set_quadrature(*q)
            if pairs is not None:
                e.set_real_pairs(pairs, 0.0)
            out.append(e.collision_step(e.phys_to_fourier(W), dt).cpu().numpy())
            e.close()
        err.append(l1rel(out[1], out[0]))
    print(f"N = {N}, {n} cells, pairs {pairs}: {np.mean(err):.3e} (bound {bound:.3e})", flush=True)
    assert np.mean(err) < bound


@pytest.mark.parametrize("N,n,J,M,Nx,kmax,bound", [(64, 300, 20, 10, 512, 4, 1.912e-10), (32, 400, 32, 16, 512, 4, 2.072e-10),
                                                   (128, 48, 16, 8, 2048, 8, 4.248e-11)])
def test_fp32_strang_step_error(N, n, J, M, Nx, kmax, bound):
    """L2 error of conserved Strang steps with one term range per cell (many cells), six states."""
    q = qbf.quadrature(N, J, wl.L_BOX, wl.R_BALL, M)
    h, dt = 1 / Nx, wl.cfl_dt(64, Nx)
    es = []
    for prec in (qbf.FP64, qbf.FP32):
        es.append(qbf.Engine(N, prec, max_cells=n))
        es[-1].set_quadrature(*q)
        es[-1].set_moment_correction(qbf.CONS_ALL)
    err = []
    for seed in range(5, 11):
        W = torch.from_numpy(wl.periodic(N, n, seed=seed, kmax=kmax)).cuda()
        a, b = (e.inhom_step_periodic(W, wl.L_BOX, h, dt) for e in es)
        err.append(float((a - b).norm() / a.norm()))
    for e in es:
        e.close()
    print(f"N = {N}, {n} cells: {np.mean(err):.3e} (bound {bound:.3e})", flush=True)
    assert np.mean(err) < bound
