"""Forward projection by lines inside an iteration (small stacks of slices)
against the FP64 oracle, over the sizes where its tables, halves and waves
end; a batch must give the same bits."""
import numpy as np
import pytest

from oracle import tgv_oracle as O
from tests.helpers import angles_deg, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SPECIAL = np.array([0.0, np.pi / 4, np.pi / 2, 3 * np.pi / 4, np.pi, -0.3, 2.0, 0.7853])
CASES = [
    # (nx, ny, nd, angles, channels, slices, detector width, detector shift)
    (80, 80, 80, angles_deg(-70, 70, 20), 1, 1, 1.0, 0.0),      # the smallest; ends on a block
    (81, 83, 120, SPECIAL, 2, 1, 1.0, 0.0),                     # ragged lines, diagonal rays
    (79, 97, 33, SPECIAL, 1, 1, 1.0, 0.0),                      # detector inside the image
    (150, 64, 300, angles_deg(-75, 75, 31), 3, 1, 1.0, 2.25),   # shifted, wider than the image
    (97, 130, 97, angles_deg(-80, 80, 33), 1, 5, 1.0, 0.0),     # slice groups 4 + 1
    (128, 129, 183, angles_deg(-70, 70, 90), 7, 9, 1.0, 0.0),   # 63 slices
    (183, 183, 259, angles_deg(-72, 72, 7), 2, 1, 1.0, 0.0),    # few angles: fewer slices a group
    (300, 410, 509, SPECIAL, 1, 1, 1.0, 0.0),                   # more than 8 waves of items
    (700, 40, 702, SPECIAL, 1, 1, 1.0, 0.0),                    # the most waves
    (96, 96, 150, SPECIAL, 1, 1, 0.6, 0.0),                     # narrow bins: gathered instead
]
# A bin sums at most 2 max(nx, ny) pixels with hat weights; in FP32 a sum of n
# positive terms taken in order is off by about sqrt(n) 2^-24, 2e-6 for 700
# lines, and the projector's own bar over these sizes is 1e-5.
BAR = 1e-5


def _problem(case):
    from graptor_amd.projector import RadonGeometry
    from graptor_amd.solver import TgvProblem
    nx, ny, nd, ang, C, nz, width, shift = CASES[case]
    g = RadonGeometry((nx, ny), ang, n_detectors=nd, detector_width=width, detector_shift=shift)
    rng = np.random.default_rng(300 + case)
    u0 = rng.random((C, nz, ny, nx)).astype(np.float32)
    f = rng.random((C, nz, g.na, nd)).astype(np.float32)
    prob = TgvProblem(f, g, (4.0, 1.0), [1.0] * C, dim=2 if nz == 1 else 3, L=30.0, u0=u0)
    return prob, u0


@pytest.mark.parametrize("case", range(len(CASES)))
def test_first_iteration_projects_the_start_image(case):
    print(f"by lines: {CASES[case][:3]}", flush=True)
    prob, u0 = _problem(case)
    prob.iterate(1, ku_on_last=True)
    got = prob.ku.cpu().numpy()
    want = O.radon_fwd(u0.astype(np.float64), prob.geometry.ofs.T, prob.nd)
    assert rel(got, want) <= BAR, rel(got, want)


def test_batch_gives_the_bits_of_each_problem():
    from graptor_amd.batch import BatchPlan
    alone = [_problem(c)[0] for c in range(len(CASES))]
    mixed = [_problem(c)[0] for c in range(len(CASES))]
    for p in alone:
        p.iterate(2, ku_on_last=True)
    BatchPlan(mixed).iterate(2, ku_on_last=True)
    for c, (a, b) in enumerate(zip(alone, mixed)):
        assert torch.equal(a.ku, b.ku), CASES[c][:3]
        assert torch.equal(a.u, b.u), CASES[c][:3]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_projection_with_scratch(case):
    """The same cases outside an iteration; the image is left alone."""
    from graptor_amd import _lib, radon
    prob, u0 = _problem(case)
    g, nx, ny, nd = prob.geometry, *CASES[case][:3]
    S = u0.shape[0] * u0.shape[1]
    img = torch.as_tensor(u0, device="cuda").reshape(S, ny, nx)
    sino = torch.empty((S, g.na, nd), device="cuda")
    radon(sino, img, (g, (nx, ny), (nd, g.na)))
    want = O.radon_fwd(u0.astype(np.float64), g.ofs.T, nd).reshape(S, g.na, nd)
    assert rel(sino.cpu().numpy(), want) <= BAR
    assert np.array_equal(img.cpu().numpy().reshape(u0.shape), u0)
    n = _lib.load().gr_radon_scratch_floats(g.handle, S)
    assert n in (0, S * nx * ny)
    assert _lib.load().gr_radon_scratch(g.handle, sino.data_ptr(), img.data_ptr(), S,
                                        img.data_ptr(), 0, None) == _lib.GR_ERR_INVALID


@pytest.mark.parametrize("C,nz,reg", [(3, 8, "TGV"), (1, 33, "TV"), (4, 12, "TGV")])
def test_slabs_of_a_small_volume_give_its_bits(C, nz, reg):
    """Whole: by lines (24 slices, with the u half of the primal step behind the
    backprojection; 33 slices) and by the gather (48 are too many for 96 x 96)."""
    from graptor_amd.projector import RadonGeometry
    from graptor_amd.slabs import SlabSolve
    from graptor_amd.solver import TgvProblem
    print(f"slabs of {C} x {nz}", flush=True)
    g = RadonGeometry((96, 96), angles_deg(-70, 70, 40), n_detectors=96)
    f = np.random.default_rng(nz).random((C, nz, 40, 96)).astype(np.float32)
    kw = dict(coupling="frobenius", discrepancy="KL", regularisation=reg, L=40.0)
    whole = TgvProblem(f, g, (4.0, 1.0), [1.0] * C, dim=3, **kw)
    parts = SlabSolve(f, g, (4.0, 1.0), [1.0] * C, 3, **kw)
    whole.iterate(6)
    parts.iterate(6)
    for name in ("u", "v", "lam", "ktl"):
        assert torch.equal(getattr(whole, name), parts.gather(name)), name
