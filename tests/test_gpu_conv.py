"""The surrogate's convolutions where their paths and splits change: dilations whose rows are staged in classes (1 to
15 at 64 x 64, odd ones among them), dilation 16 and dilated 128 x 128 images (global loads), and more blocks of rows
than workgroups (uneven ranges of blocks per workgroup).

Against the oracle with the bound of the other network tests, 1e-2 relative L2 (bfloat16 activations that round to
the neighbouring value; a wrong row, tap or channel is an error of order 1).  The result of an image does not depend
on the batch: the same sums in the same order, equal bit for bit."""
import numpy as np
import pytest

from oracle import cnn_ref as R

pytestmark = pytest.mark.gpu


def _params(seed, norm):
    rng = np.random.default_rng(seed)
    p = R.init_params(seed, cin0=5 if norm else 4)
    n = R.cout(R.NL - 1) * (9 * R.cin(R.NL - 1) + 1)
    p[-n:-R.cout(R.NL - 1)] *= 10
    return p.astype(np.float32), rng


@pytest.mark.parametrize("S", [64, 128])
@pytest.mark.parametrize("dil,norm", [((2, 3, 4, 6, 8, 1), False), ((12, 5, 16, 15, 1, 8), True), ((16, 1, 2, 7, 9, 16), False)])
def test_dilated_layers_match_oracle(S, dil, norm):
    import torch
    from qbf.cnn import CNN
    p, rng = _params(sum(dil), norm)
    x = (0.5 * rng.standard_normal((2, 4, S, S))).astype(np.float32)
    t = (0.3 * rng.standard_normal((2, 4, S, S))).astype(np.float32)
    net = CNN(max_batch=2, params=p, N=S, dil=dil, norm=norm)
    out = net.forward(torch.from_numpy(x).cuda()).cpu().numpy()
    ref, _ = R.forward(x, p, dil=dil, norm=norm, bf16_round=True)
    e = np.linalg.norm(out - ref) / np.linalg.norm(ref)
    net.gradients(torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda())
    g = net.get_params(grads=True)
    net.close()
    _, gref, _ = R.gradients(x, t, p, dil=dil, norm=norm, bf16_round=True)
    eg = np.linalg.norm(g - gref) / np.linalg.norm(gref)
    print(f"S = {S}, dil = {dil}: forward {e:.2e}, gradients {eg:.2e}", flush=True)
    assert e < 1e-2 and eg < 2e-2


@pytest.mark.parametrize("S,B", [(64, 33), (64, 70), (128, 17), (128, 35)])
@pytest.mark.parametrize("dil", [(1,) * 6, (3, 2, 1, 16, 4, 6)])
def test_images_do_not_depend_on_the_batch(S, B, dil):
    import torch
    from qbf.cnn import CNN
    p, rng = _params(S + B, False)
    x = torch.from_numpy((0.5 * rng.standard_normal((B, 4, S, S))).astype(np.float32)).cuda()
    net = CNN(max_batch=B, params=p, N=S, dil=dil)
    y = net.forward(x).clone()
    for b in (0, 1, B // 2, B - 2, B - 1):
        assert torch.equal(net.forward(x[b:b + 1].contiguous())[0], y[b]), b
    net.close()
