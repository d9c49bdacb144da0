"""The convolutions' two taps per MFMA and the tap left over: every output-channel blocking on planes
smaller than, equal to and one beyond a tile, against the CPU oracle with the other convolution tests'
bound (the output's BF16 rounding, 2^-8 of it, and 2e-5 of the sum of the terms' magnitudes), and the
same bits on every call, of the convolutions and of a whole prediction (its layers chain MFMAs on one
accumulator).
"""
import numpy as np
import pytest

from oracle import unet3d as U

pytestmark = pytest.mark.gpu


def _bits(torch, a):
    return torch.from_numpy(U.bf16_bits(a).view(np.int16)).cuda()


@pytest.mark.parametrize("D,H,W,C,Cout", [(1, 1, 1, 16, 16), (2, 8, 64, 16, 16), (2, 9, 65, 32, 16), (1, 4, 64, 16, 32),
                                          (2, 5, 65, 16, 48), (3, 3, 30, 32, 64), (1, 5, 66, 16, 128)])
def test_conv_forward(pkg, gpu_available, D, H, W, C, Cout):
    import torch
    rng = np.random.default_rng(100 * H + W + Cout)
    x = U.bf16(rng.normal(size=(D, H, W, C)))
    w = U.bf16(0.1 * rng.normal(size=(27, Cout, C)))
    xb, wb = _bits(torch, x), _bits(torch, w)
    outs = [pkg.conv3d_bf16_forward(xb, wb).clone() for _ in range(3)]
    assert all(torch.equal(outs[0], o) for o in outs)
    got = U.from_bits(outs[0].cpu().numpy().view(np.uint16))
    exact, mag = U.conv(x, w), U.conv(np.abs(x), np.abs(w))
    assert np.all(np.abs(got - exact) <= 2.0 ** -8 * np.abs(exact) + 2e-5 * mag)


@pytest.mark.parametrize("shape", [(16, 64, 64), (8, 72, 136)])
def test_prediction_is_the_same_every_time(pkg, gpu_available, shape):
    import torch
    torch.manual_seed(1)
    v = torch.randn(shape, dtype=torch.complex64, device="cuda")
    with pkg.WarmStartNet(*shape, seed=3) as net:
        outs = [torch.view_as_real(net.predict(v).clone()) for _ in range(5)]
        torch.cuda.synchronize()
    assert all(torch.equal(outs[0], o) for o in outs)
