"""The identity behind the mirrored I3 terms (csrc/qbf_i3fold.hip), in numpy on the CPU, and which
terms the quadrature tables pair.

For a term with psi1 = E (a translation phase) and its mirror (conj(E), the same psi2), CdInt's sum
over both follows from the products K[S_i .* F_j] of the first alone."""
import numpy as np
import pytest

import oracle as O


def pad(x):
    N = x.shape[-1]
    i = np.r_[0:N // 2, 2 * N - N // 2:2 * N]
    y = np.zeros(x.shape[:-2] + (2 * N, 2 * N), np.complex128)
    y[..., i[:, None], i] = x
    return y


def extract(y):
    N = y.shape[-1] // 2
    i = np.r_[0:N // 2, 2 * N - N // 2:2 * N]
    return y[..., i[:, None], i]


F, IF = np.fft.fft2, np.fft.ifft2


@pytest.mark.parametrize("N,J,M", [(4, 2, 2), (8, 4, 3), (8, 2, 4), (16, 2, 5)])
def test_mirror_identity(N, J, M):
    rng = np.random.default_rng(N + M)
    # complex spectra with content on the Nyquist lines: nothing may rest on W being Hermitian
    W = rng.standard_normal((4, N, N)) + 1j * rng.standard_normal((4, N, N))
    p1, p2 = O.fourier_I3(N, J, 6.0, 3.75, M)
    p1 = p1.reshape(J, M, N, N)
    p2 = p2.reshape(J, M, 2 * N, 2 * N)
    eta = np.array([1.0, -1, -1, -1])
    S = F(pad(W))

    def direct(psi1, psi2):
        Fq = F(pad(psi1 * W))
        return np.stack([extract(IF(sum(eta[i] * Fq[i] * F(psi2 * IF(S[i] * Fq[j])) for i in range(4)))) for j in range(4)])

    for j in range(J):
        for m in range(M // 2):
            # the Gauss-Legendre nodes m and M - 1 - m are +-rho with equal weights
            a, b = p1[j, m], p1[j, M - 1 - m]
            assert np.abs(a - b.conj()).max() < 4e-13
            assert np.abs(p2[j, m] - p2[j, M - 1 - m]).max() < 4e-13 * np.abs(p2[j, m]).max()
            Fq = F(pad(a * W))
            Y = np.array([[F(p2[j, m] * IF(S[i] * Fq[k])) for k in range(4)] for i in range(4)])
            out = np.stack([extract(IF((eta[:, None, None] * Fq * Y[:, k]).sum(0))) for k in range(4)])
            out += a.conj() * np.stack([extract(IF((eta[:, None, None] * S * Y[i]).sum(0))) for i in range(4)])
            ref = direct(a, p2[j, m]) + direct(b, p2[j, M - 1 - m])
            assert np.abs(out - ref).sum() < 1e-12 * np.abs(ref).sum()
