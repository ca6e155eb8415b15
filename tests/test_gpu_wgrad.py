"""Weight and bias gradients of the surrogate where their split changes: rows per workgroup (4, 8, 16, by the
number of images), one or two 64-pixel segments per row, staging with and without dilation.

The loss is a mean, so the gradients of B images are the mean of the gradients of the images taken alone.  For B
a power of two the factor 1 / B is exact in bfloat16, so both sides sum the same products in fp32: n = B S^2 terms
of random sign, error about 2^-24 sqrt(n) of the sum, 4e-5 at the largest.  1e-4 relative L2 is allowed; a row or a
tap that is missing or taken twice is an error of 1e-2 or more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,B", [(64, 2), (64, 32), (64, 64), (128, 8), (128, 16)])
@pytest.mark.parametrize("dil", [(1,) * 6, (1, 2, 4, 8, 4, 1)])
def test_batch_gradients_are_the_mean_of_single_image_gradients(S, B, dil):
    import torch
    from qbf.cnn import CNN
    rng = np.random.default_rng(S + B)
    x = torch.from_numpy((0.5 * rng.standard_normal((B, 4, S, S))).astype(np.float32)).cuda()
    t = torch.from_numpy((0.3 * rng.standard_normal((B, 4, S, S))).astype(np.float32)).cuda()
    net = CNN(max_batch=B, N=S, dil=dil)
    net.gradients(x, t)
    g = net.get_params(grads=True).astype(np.float64)
    one = np.zeros_like(g)
    for b in range(B):
        net.gradients(x[b:b + 1].contiguous(), t[b:b + 1].contiguous())
        one += net.get_params(grads=True).astype(np.float64) / B
    net.close()
    e = np.linalg.norm(g - one) / np.linalg.norm(one)
    print(f"S = {S}, B = {B}, dil = {dil}: {e:.2e}", flush=True)
    assert e < 1e-4
