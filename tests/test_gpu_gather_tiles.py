"""The two kernels that large stacks take, at sizes the oracle can follow: the
gather of the forward projection (gr_radon, which never projects by lines) and
the tiles of the backprojection (images with too many rows of waves to be read
directly)."""
import numpy as np
import pytest

from oracle import tgv_oracle as O
from tests.helpers import angles_deg, rel
from tests.test_gpu_projector import CASES

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

BAR = 1e-5  # the projector's own bar


def _gather(g, img):
    from graptor_amd import _lib
    S = img.shape[0]
    sino = torch.empty((S, g.na, g.nd), device="cuda")
    dev = torch.as_tensor(img, device="cuda")
    _lib.check(_lib.load().gr_radon(g.handle, sino.data_ptr(), dev.data_ptr(), S,
                                    torch.cuda.current_stream().cuda_stream))
    return sino.cpu().numpy()


# the cases of the projector's tests, and a slice of the large volume's geometry
FORWARD = CASES + [(512, 512, 512, np.deg2rad(np.linspace(-75, 75, 90)) + np.pi / 2, 3)]


@pytest.mark.parametrize("case", range(len(FORWARD)))
def test_gather_matches_oracle(case):
    from graptor_amd.projector import RadonGeometry
    nx, ny, nd, ang, ns = FORWARD[case]
    print(f"gather {nx}x{ny} nd={nd} na={ang.size} slices={ns}", flush=True)
    g = RadonGeometry((nx, ny), ang, n_detectors=nd)
    img = np.random.default_rng(100 + case).random((ns, ny, nx)).astype(np.float32)
    want = O.radon_fwd(img.astype(np.float64), g.ofs.T.copy(), nd)
    assert rel(_gather(g, img), want) <= BAR


@pytest.mark.parametrize("band", [4, 8, 16, 32])
@pytest.mark.parametrize("ns", [1, 2, 4])
def test_gather_bands(band, ns):
    from graptor_amd.projector import RadonGeometry
    print(f"gather bands of {band}, {ns} slices", flush=True)
    g = RadonGeometry((100, 97), angles_deg(-75, 75, 25), n_detectors=110)
    g.set_tuning(fwd_band=band)
    img = np.random.default_rng(11).random((ns, 97, 100)).astype(np.float32)
    want = O.radon_fwd(img.astype(np.float64), g.ofs.T.copy(), 110)
    assert rel(_gather(g, img), want) <= BAR


@pytest.mark.parametrize("tile", [4, 8, 16, 32])
@pytest.mark.parametrize("ns", [1, 2, 3, 8, 11])
def test_tiles_match_oracle(ns, tile):
    """13 x 515 rows of 64 pixels are more than the 6144 waves up to which bins
    are read directly, whatever the slices per wave.  Tiles of up to 16 rows
    have four accumulator rows a lane and, from 8 slices on, groups of eight."""
    from graptor_amd import radon_ad
    from graptor_amd.projector import RadonGeometry
    print(f"tiles of {tile} rows, {ns} slices", flush=True)
    nx, ny, nd, na = 810, 515, 400, 9
    g = RadonGeometry((nx, ny), angles_deg(-80, 85, na), n_detectors=nd)
    g.set_tuning(adj_tile_y=tile)
    sino = np.random.default_rng(12 + ns).random((ns, na, nd)).astype(np.float32)
    back = torch.empty((ns, ny, nx), device="cuda")
    radon_ad(back, torch.as_tensor(sino, device="cuda"), g)
    want = O.radon_adj(sino.astype(np.float64), g.ofs.T.copy(), nx, ny)
    assert rel(back.cpu().numpy(), want) <= BAR
