"""The FP64 operator-norm rounds against the FP64 oracle at the edges of their
tiles: fewer bins than a wave, ragged images, more tiles than partial sums."""
import numpy as np
import pytest

from oracle import tgv_oracle as O
from tests.helpers import angles_deg

pytestmark = pytest.mark.gpu

pytest.importorskip("torch")

# Both sides sum a few thousand FP64 terms per value, in different orders:
# 1e-16 sqrt(1e4) a round, ten rounds.
BAR = 1e-12


@pytest.mark.parametrize("nx,ny,nd,na", [(5, 3, 7, 4), (16, 16, 64, 5), (17, 31, 65, 9),
                                         (130, 47, 129, 33), (523, 530, 90, 3)])
def test_normest_rounds(nx, ny, nd, na):
    from graptor_amd import radon_normest
    from graptor_amd.projector import RadonGeometry
    print(f"normest {nx}x{ny} nd={nd} na={na}", flush=True)
    g = RadonGeometry((nx, ny), angles_deg(-80, 100, na), n_detectors=nd)
    ofs = g.ofs.T.copy()
    x0 = np.random.default_rng(nx).random((nx, ny))
    got = radon_normest(None, g, mode="reference", x0=x0, iters=10)
    want = O.normest_reference(ofs, nx, ny, nd, x0.T, iters=10)
    assert abs(got - want) <= BAR * abs(want), (got, want)
    # a fixed number of power rounds from the same start
    got = radon_normest(None, g, mode="power", x0=x0, iters=6, tol=0.0)
    x = x0.T.copy()
    for _ in range(6):
        x = x / np.linalg.norm(x)
        y = O.radon_adj(O.radon_fwd(x, ofs, nd), ofs, nx, ny)
        lam = float((x * y).sum())
        x = y
    assert abs(got - np.sqrt(lam)) <= BAR * abs(got), (got, np.sqrt(lam))
