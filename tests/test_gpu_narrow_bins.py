"""Detector bins narrower than a pixel against the FP64 oracle: the shadow of a
backprojection tile covers more of them than of unit bins.  Small stacks (read
directly), tiles of every height and slice group, batches, the fused primal
step, and bins too narrow for any tile."""
import numpy as np
import pytest

from oracle import tgv_oracle as O
from tests.helpers import angles_deg, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _bar(width):
    # positions in FP32 are off by some 2^-24 of their number of bins: the bar
    # of unit bins, scaled with the bins per pixel
    return 1e-5 / width


def _geometry(nx, ny, na, width, nd=None):
    from graptor_amd.projector import RadonGeometry
    nd = nd or int(0.8 * max(nx, ny) / width)
    return RadonGeometry((nx, ny), angles_deg(-80, 85, na), n_detectors=nd, detector_width=width)


def _check(g, S, seed):
    from graptor_amd import radon_ad
    nx, ny = g.shape
    sino = np.random.default_rng(seed).random((S, g.na, g.nd)).astype(np.float32)
    back = torch.empty((S, ny, nx), device="cuda")
    radon_ad(back, torch.as_tensor(sino, device="cuda"), g)
    want = O.radon_adj(sino.astype(np.float64), g.ofs.T.copy(), nx, ny)
    return rel(back.cpu().numpy(), want)


@pytest.mark.parametrize("width", [0.97, 0.6, 0.25, 0.04])
@pytest.mark.parametrize("S", [1, 5])
def test_small_stacks(S, width):
    print(f"narrow {width} {S} small", flush=True)
    assert _check(_geometry(97, 90, 17, width), S, 1) <= _bar(width)


@pytest.mark.parametrize("width", [0.97, 0.6, 0.25])
@pytest.mark.parametrize("S,tile", [(1, 16), (2, 32), (3, 8), (9, 16), (4, 4), (9, 32)])
def test_tiles(S, tile, width):
    """13 x 515 rows of 64 pixels are too many to be read directly."""
    print(f"narrow {width} {S} tiles of {tile}", flush=True)
    g = _geometry(810, 515, 7, width, nd=700)
    g.set_tuning(adj_tile_y=tile)
    assert _check(g, S, 2) <= _bar(width)


@pytest.mark.parametrize("S", [1, 9])
def test_bins_too_narrow_for_tiles(S):
    """One angle's shadow of a tile is 65000 bins."""
    width = 0.001
    print(f"narrow {width} {S}", flush=True)
    assert _check(_geometry(810, 515, 2, width, nd=2000), S, 3) <= _bar(width)


@pytest.mark.parametrize("width", [0.97, 0.6, 0.25])
def test_batch_and_fused_primal_step(width):
    from graptor_amd.batch import BatchPlan
    from graptor_amd.solver import TgvProblem
    print(f"narrow {width} batch", flush=True)

    def problem(fuse):
        g = _geometry(81, 81, 15, width)
        g.set_fusion(fuse)
        f = np.random.default_rng(5).random((3, 1, g.na, g.nd)).astype(np.float32)
        return TgvProblem(f, g, (4.0, 1.0), [1.0, 0.5, 0.2], dim=2, discrepancy="L2", L=30.0)

    alone, batch, fused, fused_batch = problem(False), problem(False), problem(True), problem(True)
    alone.iterate(3)
    BatchPlan([batch]).iterate(3)
    fused.iterate(3)
    BatchPlan([fused_batch]).iterate(3)
    want = O.radon_adj(alone.lam.cpu().numpy().astype(np.float64), alone.geometry.ofs.T.copy(),
                       81, 81)
    assert rel(alone.ktl.cpu().numpy(), want) <= _bar(width)
    u = alone.u.cpu().numpy()
    assert np.abs(u).sum() > 0
    for other in (batch, fused, fused_batch):
        assert rel(other.u.cpu().numpy(), u) <= 1e-6


def test_too_narrow_for_batches_and_fusion_is_refused():
    from graptor_amd.batch import BatchPlan
    from graptor_amd.solver import TgvProblem
    g = _geometry(40, 40, 3, 0.001, nd=50)
    f = np.ones((1, 1, 3, 50), np.float32)
    prob = TgvProblem(f, g, (4.0, 1.0), [1.0], dim=2, coupling="uncorrelated", L=30.0)
    prob.iterate(1)
    with pytest.raises(ValueError, match="too narrow"):
        BatchPlan([prob])
    g.set_fusion(True)
    with pytest.raises(ValueError, match="too narrow"):
        prob.iterate(1)
