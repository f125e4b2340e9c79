"""Weight gradients at the edges of the kernel's tiles: ragged widths around
its segments of 32 and 64 pixels, channels short of a tile, walks of one and of
many rows, channel slices."""
import numpy as np
import pytest
import torch

from oracle import cnn_oracle as orc
from tests.test_gpu_cnn import bf16_round, chk, lib, rel, stream, to_dev_bf16

pytestmark = pytest.mark.gpu

CASES = [
    # (taps, cin, cout, n, H, W)
    (9, 8, 8, 1, 1, 1),          # one pixel
    (9, 16, 40, 1, 3, 31),       # within a segment of 32; part of a tile each way
    (9, 32, 32, 2, 5, 33),       # 33 pixels: a segment of 64
    (9, 40, 32, 1, 4, 64),       # a whole segment
    (9, 24, 72, 2, 2, 65),       # one pixel in the second segment
    (9, 32, 32, 9, 90, 129),     # walks of more than one row, three segments
    (9, 64, 32, 40, 31, 20),     # and with segments of 32
    (1, 16, 8, 2, 3, 63),
    (1, 40, 64, 5, 60, 130),
]


@pytest.mark.parametrize("taps,cin,cout,n,H,W", CASES)
def test_weight_gradient(taps, cin, cout, n, H, W):
    print(f"wgrad {taps} {cin}->{cout} {n} x {H} x {W}", flush=True)
    rng = np.random.default_rng(cin + cout + W)
    x = bf16_round(rng.standard_normal((n, H, W, cin + 16)))
    dy = bf16_round(rng.standard_normal((n, H, W, cout + 8)))
    xd, dyd = to_dev_bf16(x), to_dev_bf16(dy)
    dw = torch.ones(cout * taps * cin + 1, device="cuda")
    chk(lib().gr_cnn_conv_wgrad(xd.data_ptr(), cin + 16, 8, dyd.data_ptr(), cout + 8, 8,
                                dw.data_ptr(), n, H, W, cin, cout, taps, 1, stream()))
    got = dw.cpu().double().numpy()
    assert got[-1] == 1.0
    w = np.zeros((cout, taps, cin))
    ref = 1.0 + orc.conv_backward(x[..., 8:8 + cin], w, dy[..., 8:])[1]
    # FP32 sums of exact products, as for the other weight gradients
    assert rel(got[:-1].reshape(cout, taps, cin), ref) < 2e-6
