"""Detector bins wider than a pixel, whose hats reach over more pixels of a line
than unit bins' do, against the FP64 oracle: projections alone, in iterations
and in batches, the feasibility mask and the operator norm.  1.06 pixels are
the most that three candidates hold."""
import numpy as np
import pytest

from oracle import tgv_oracle as O
from tests.helpers import angles_deg, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SPECIAL = np.array([0.0, np.pi / 4, np.pi / 2, 3 * np.pi / 4, np.pi, -0.3, 2.0, 0.7853])
CASES = [
    # (nx, ny, nd, angles, slices, detector width)
    (64, 64, 64, angles_deg(-70, 70, 20), 1, 1.05),
    (64, 64, 60, SPECIAL, 2, 1.07),
    (100, 97, 80, angles_deg(-75, 75, 25), 5, 1.5),
    (81, 130, 90, SPECIAL, 3, 1.6),
    (96, 96, 50, angles_deg(-80, 80, 31), 9, 2.0),
    (40, 33, 30, SPECIAL, 1, 3.7),
    (90, 90, 21, angles_deg(0, 180, 12), 2, 40.0),  # a bin holds half the image
    (30, 30, 12, SPECIAL, 1, 100.0),                # and all of it
]
# FP32 sums of positive terms in order: sqrt(n) 2^-24, 5e-6 for the 8000 pixels
# of the widest bins; the projector's own bar
BAR = 1e-5


def _geometry(case):
    from graptor_amd.projector import RadonGeometry
    nx, ny, nd, ang, S, width = CASES[case]
    return RadonGeometry((nx, ny), ang, n_detectors=nd, detector_width=width)


def _problem(case):
    from graptor_amd.solver import TgvProblem
    nx, ny, nd, ang, S, width = CASES[case]
    g = _geometry(case)
    rng = np.random.default_rng(700 + case)
    u0 = rng.random((S, 1, ny, nx)).astype(np.float32)
    f = rng.random((S, 1, g.na, nd)).astype(np.float32)
    return TgvProblem(f, g, (4.0, 1.0), [1.0] * S, dim=2, L=100.0, u0=u0), u0


@pytest.mark.parametrize("case", range(len(CASES)))
def test_projection(case):
    from graptor_amd import radon
    print(f"wide bins {CASES[case][:3]} {CASES[case][-1]}", flush=True)
    prob, u0 = _problem(case)
    g, S = prob.geometry, u0.shape[0]
    want = O.radon_fwd(u0.astype(np.float64), g.ofs.T, g.nd)
    sino = torch.empty((S, 1, g.na, g.nd), device="cuda")
    radon(sino, torch.as_tensor(u0, device="cuda"), g)
    assert rel(sino.cpu().numpy(), want) <= BAR
    prob.iterate(1, ku_on_last=True)
    assert rel(prob.ku.cpu().numpy(), want) <= BAR


def test_batch():
    from graptor_amd.batch import BatchPlan
    probs, u0 = zip(*[_problem(c) for c in range(len(CASES))])
    BatchPlan(probs).iterate(1, ku_on_last=True)
    for c, (p, u) in enumerate(zip(probs, u0)):
        want = O.radon_fwd(u.astype(np.float64), p.geometry.ofs.T, p.nd)
        assert rel(p.ku.cpu().numpy(), want) <= BAR, CASES[c]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_operator_norm_and_mask(case):
    from graptor_amd import make_function_feasible, radon_normest
    nx, ny, nd, ang, S, width = CASES[case]
    g = _geometry(case)
    ofs = g.ofs.T.copy()
    x0 = np.random.default_rng(case).random((nx, ny))
    got = radon_normest(None, g, mode="reference", x0=x0, iters=5)
    want = O.normest_reference(ofs, nx, ny, nd, x0.T, iters=5)
    # a few thousand FP64 terms per value on both sides
    assert abs(got - want) <= 1e-12 * abs(want), (got, want)
    f = torch.ones((1, g.na, nd), device="cuda")
    make_function_feasible(f, g)
    reached = O.radon_fwd(np.ones((ny, nx)), ofs, nd)
    # bins that FP32 positions cannot tell from empty ones are left open
    open_ = (reached > 0) & (reached < 1e-3)
    kept = f[0].cpu().numpy() > 0
    assert np.array_equal(kept[~open_], (reached > 0)[~open_])
