"""Backprojection of small stacks, read directly, against the FP64 oracle and,
bit for bit, against the slices of a stack large enough for the tile kernel."""
import numpy as np
import pytest

from oracle import tgv_oracle as O
from tests.helpers import angles_deg, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

CASES = [
    # (nx, ny, nd, angles, slices of the small stack, slices of the large one)
    (5, 3, 7, 4, 1, 2100),                 # a corner of one tile
    (64, 16, 64, 20, 4, 2052),             # exactly a tile; one slice a wave
    (65, 18, 50, 257, 2, 1030),            # ragged; one angle beyond a chunk of the table
    (183, 183, 183, 31, 11, 63),           # 6039 waves of one slice
    (183, 183, 120, 31, 13, 63),           # two a wave, the last pair half empty
    (256, 255, 363, 12, 23, 45),           # four a wave, the last group of three
    (300, 270, 270, 9, 5, 25),             # tiles of 32 rows
]


@pytest.mark.parametrize("nx,ny,nd,na,few,many", CASES)
def test_small_stacks_backproject_like_large_ones(nx, ny, nd, na, few, many):
    from graptor_amd import radon_ad
    from graptor_amd.projector import RadonGeometry
    print(f"direct {nx}x{ny} nd={nd} na={na} slices={few}", flush=True)
    g = RadonGeometry((nx, ny), angles_deg(-80, 85, na), n_detectors=nd)
    rs = (g, (nx, ny), (nd, na))
    gen = torch.Generator(device="cuda").manual_seed(nx + few)
    sino = torch.rand((many, na, nd), device="cuda", generator=gen) - 0.5
    small = torch.empty((few, ny, nx), device="cuda")
    large = torch.empty((many, ny, nx), device="cuda")
    radon_ad(small, sino[:few].clone(), rs)
    radon_ad(large, sino, rs)
    assert torch.equal(small, large[:few])
    want = O.radon_adj(sino[:few].cpu().numpy().astype(np.float64), g.ofs.T.copy(), nx, ny)
    # the projector's own bar: positions in FP32 are off by up to nd 2^-24 of a bin
    assert rel(small.cpu().numpy(), want) <= 1e-5
