"""gr_radon_scratch refuses scratch that shares memory with its image or its
sinogram, where it would be used."""
import pytest

from oracle import tgv_oracle as O
from tests.helpers import angles_deg, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("of_slices", [0, 3])
def test_scratch_overlaps(of_slices):
    from graptor_amd import _lib
    from graptor_amd.projector import RadonGeometry
    N, na, S = 90, 20, 2
    g = RadonGeometry((N, N), angles_deg(-70, 70, na), n_detectors=N)
    n, m = S * N * N, S * na * N
    assert _lib.load().gr_radon_scratch_floats(g.handle, S) == n
    # one array: scratch-sized room, image, scratch-sized room, sinogram, room
    mem = torch.zeros(3 * n + m + n, device="cuda")
    img, sino = mem[n:2 * n], mem[3 * n:3 * n + m]
    img.copy_(torch.rand(n, generator=torch.Generator().manual_seed(1)))
    want = O.radon_fwd(img.view(S, N, N).double().cpu().numpy(), g.ofs.T.copy(), N)

    def run(at):
        return _lib.load().gr_radon_scratch(
            g.handle, sino.data_ptr(), img.data_ptr(), S, mem[at:].data_ptr(), of_slices,
            torch.cuda.current_stream().cuda_stream)

    for at in (1, n, 2 * n - 1, 2 * n + 1, 3 * n, 3 * n + m - 1):
        assert run(at) == _lib.GR_ERR_INVALID, at
        assert float(sino.abs().sum()) == 0.0
    for at in (0, 2 * n, 3 * n + m):  # right beside them
        sino.zero_()
        assert run(at) == _lib.GR_OK, at
        assert rel(sino.view(S, na, N).cpu().numpy(), want) <= 1e-5
