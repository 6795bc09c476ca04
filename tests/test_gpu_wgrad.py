"""The weight and bias gradients of the convolutions (k_conv_wgrad) at the edges of their
tiles: rows that fill, start and overrun a K step of 32, 16 and 8 voxels, y and z tile
remainders, several spatial tiles per block, eight input channels, and tensors that are
only 2-byte aligned.

x and dz are BF16, the products are exact in FP32 and only their sum rounds: against the
FP64 sum each of the N terms adds at most one rounding of 2^-24 of the running sum, so
|error| <= N 2^-24 sum|x dz| per element.
"""
import numpy as np
import pytest

from oracle import unet_oracle as U

pytestmark = pytest.mark.gpu

CASES = [((1, 1, 1), 8, 16), ((4, 4, 32), 16, 16), ((5, 3, 33), 16, 32), ((9, 9, 16), 8, 16), ((3, 10, 17), 32, 16),
         ((8, 8, 8), 64, 128), ((9, 5, 7), 16, 16), ((5, 9, 40), 48, 16), ((2, 6, 24), 24, 48), ((9, 17, 40), 192, 64),
         ((20, 37, 70), 16, 16)]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape,cin,cout", CASES)
def test_weight_gradient(shape, cin, cout, offset):
    import torch
    from shiokaze_amd import learned
    rng = np.random.default_rng(sum(shape) + cin)
    n = int(np.prod(shape))

    def tensor(c):
        a = U.bf16_round(rng.standard_normal(n * c))
        t = torch.zeros(n * c + offset, dtype=torch.bfloat16, device="cuda")
        t[offset:] = torch.from_numpy(a.astype(np.float32)).cuda().bfloat16()
        return a.reshape(*shape, c), t[offset:].view(*shape, c)

    x, xt = tensor(cin)
    dz, dzt = tensor(cout)
    w = torch.zeros((27, cin, cout), device="cuda")
    _, dw, db = learned.conv3d_backward(xt, w, dzt, need_dx=False)
    rw, rb = U.conv3d_wgrad(x, dz)
    bw, bb = U.conv3d_wgrad(np.abs(x), np.abs(dz))
    eps = n * 2.0 ** -24
    assert np.all(np.abs(dw.cpu().numpy() - rw) <= eps * bw + 1e-30)
    assert np.all(np.abs(db.cpu().numpy() - rb) <= eps * bb + 1e-30)
    _, dw2, db2 = learned.conv3d_backward(xt, w, dzt, need_dx=False)
    assert torch.equal(dw, dw2) and torch.equal(db, db2)   # one order of summation
