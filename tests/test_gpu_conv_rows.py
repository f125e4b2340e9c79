"""3x3 convolutions whose grids take the row kernel, at the edges of its tiles:
against the oracle, and bit for bit against single images, whose small grids
take the tile kernel."""
import numpy as np
import pytest
import torch

from oracle import cnn_oracle as orc
from tests.test_gpu_cnn import bf16_round, chk, lib, rel, stream, to_dev_bf16

pytestmark = pytest.mark.gpu

CASES = [
    # (cin, cout, H, W, n, ldy, cy0, float32 output)
    (16, 32, 9, 40, 90, 32, 0, True),      # one chunk of 16; ragged rows and pixels
    (48, 32, 8, 130, 64, 32, 0, False),    # a chunk and a half; two segments
    (32, 64, 9, 65, 43, 96, 32, False),    # channel slice of a wider buffer
    (96, 96, 4, 70, 90, 100, 4, False),    # scalar stores (unaligned slice)
    (48, 192, 4, 64, 90, 192, 0, True),    # three blocks of output channels
    (16, 128, 11, 33, 44, 128, 0, False),  # 32 pixels x 128 channels
    (32, 256, 8, 20, 70, 256, 0, True),    # two blocks of 128
    (32, 256, 6, 20, 50, 256, 0, False),   # two rows a work-group from here on
    (32, 32, 5, 40, 100, 32, 0, False),
    (16, 32, 2, 128, 256, 32, 0, True),
    (64, 64, 6, 64, 100, 64, 0, False),
]


@pytest.mark.parametrize("cin,cout,H,W,n,ldy,cy0,f32", CASES)
def test_row_convolution(cin, cout, H, W, n, ldy, cy0, f32):
    print(f"conv rows {cin}->{cout} {n} x {H} x {W}", flush=True)
    rng = np.random.default_rng(cin + cout + H)
    x = bf16_round(rng.standard_normal((n, H, W, cin)))
    w = bf16_round(rng.standard_normal((cout, 9, cin)) / np.sqrt(9 * cin))
    b = rng.standard_normal(cout).astype(np.float32)
    xd, wd, bd = to_dev_bf16(x), to_dev_bf16(w), torch.as_tensor(b).cuda()
    dt = torch.float32 if f32 else torch.bfloat16

    def run(images):
        y = torch.full((images.shape[0], H, W, ldy), 7.0, device="cuda", dtype=dt)
        chk(lib().gr_cnn_conv_fwd(images.data_ptr(), cin, 0, wd.data_ptr(), bd.data_ptr(),
                                  y.data_ptr(), ldy, cy0, images.shape[0], H, W, cin, cout, 9, 1,
                                  int(f32), stream()))
        return y

    got = run(xd)
    for i in (0, n // 2, n - 1):
        assert torch.equal(got[i], run(xd[i:i + 1])[0]), i
    rest = torch.cat([got[..., :cy0], got[..., cy0 + cout:]], dim=-1)
    assert bool((rest == 7.0).all())
    ref = orc.conv(x[[0, n - 1]], w, b.astype(np.float64), relu=True)
    out = got[[0, n - 1]][..., cy0:cy0 + cout].double().cpu().numpy()
    assert rel(out, ref) < (2e-6 if f32 else 8e-3)  # FP32 sums, bf16 output rounding
