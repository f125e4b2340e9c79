"""ReLU mask and bias gradient in one call against the two separate calls: the
mask bit for bit, the sum within FP32 summation error; vector and scalar forms,
pixel counts around the lanes of a block."""
import pytest
import torch

from tests.test_gpu_cnn import chk, lib, stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npix,c,ldd,cd0,ldy,cy0", [
    (1, 8, 8, 0, 8, 0), (63, 32, 32, 0, 96, 32), (65, 32, 64, 8, 32, 0), (70001, 64, 64, 0, 64, 0),
    (1000, 256, 256, 0, 384, 128), (500, 16, 20, 4, 16, 0), (77, 4, 4, 0, 8, 4)])
def test_relu_and_bias_gradient(npix, c, ldd, cd0, ldy, cy0):
    print(f"relu + bias {npix} x {c}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(npix + c)
    dy = torch.randn((npix, ldd), device="cuda", generator=gen).to(torch.bfloat16)
    y = torch.randn((npix, ldy), device="cuda", generator=gen).clamp_min(0).to(torch.bfloat16)
    want, got = dy.clone(), dy.clone()
    db = torch.full((2, c), 0.5, device="cuda")
    L, s = lib(), stream()
    chk(L.gr_cnn_relu_bwd(want.data_ptr(), ldd, cd0, y.data_ptr(), ldy, cy0, npix, c, s))
    chk(L.gr_cnn_bias_grad(want.data_ptr(), ldd, cd0, npix, c, db[0].data_ptr(), s))
    chk(L.gr_cnn_relu_bias_grad(got.data_ptr(), ldd, cd0, y.data_ptr(), ldy, cy0, npix, c,
                                db[1].data_ptr(), s))
    assert torch.equal(got, want)
    # a sum of n unit terms in FP32 is off by up to about sqrt(n) * sqrt(n) 2^-24
    scale = want[:, cd0:cd0 + c].float().abs().sum(0) + 0.5
    assert bool(((db[0] - db[1]).abs() <= 2e-6 * scale).all())
    with pytest.raises(ValueError):
        chk(L.gr_cnn_relu_bias_grad(got.data_ptr(), ldd, cd0, y.data_ptr(), ldy, cy0, npix, 96,
                                    db[1].data_ptr(), s))
