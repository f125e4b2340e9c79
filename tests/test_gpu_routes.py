"""Which way forward projections go, and that parts of a stack follow the whole:
by lines up to a size, by the gather above it and with the primal step fused
into the backprojection."""
import numpy as np
import pytest

from oracle import tgv_oracle as O
from tests import test_gpu_lines as lines
from tests.helpers import angles_deg, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# 128 x 129 with 63 slices and 90 angles is more than a stack by lines holds;
# bins narrower than a pixel are never projected by lines
BY_LINES = [True] * 5 + [False] + [True] * 3 + [False]


@pytest.mark.parametrize("case", range(len(BY_LINES)))
def test_cases_by_lines(case):
    from graptor_amd import _lib
    assert len(lines.CASES) == len(BY_LINES)
    nx, ny, nd, ang, C, nz, width, shift = lines.CASES[case]
    from graptor_amd.projector import RadonGeometry
    g = RadonGeometry((nx, ny), ang, n_detectors=nd, detector_width=width, detector_shift=shift)
    S = C * nz
    assert g.iterates_by_lines(S) == BY_LINES[case]
    assert _lib.load().gr_radon_scratch_floats(g.handle, S) == BY_LINES[case] * S * nx * ny


def test_four_slices_a_work_group_against_the_oracle():
    """Stacks with enough angles and slices for groups of four: an iteration and
    a projection alone."""
    from graptor_amd import _lib, radon
    from graptor_amd.projector import RadonGeometry
    from graptor_amd.solver import TgvProblem
    nx, ny, nd, na, C, nz = 160, 161, 228, 64, 5, 4  # 320 work-groups
    print(f"lines {nx}x{ny}x{C * nz}", flush=True)
    g = RadonGeometry((nx, ny), angles_deg(-80, 80, na), n_detectors=nd)
    assert g.iterates_by_lines(C * nz)
    assert _lib.load().gr_radon_scratch_floats(g.handle, C * nz) == C * nz * nx * ny
    rng = np.random.default_rng(4)
    u0 = rng.random((C, nz, ny, nx)).astype(np.float32)
    f = rng.random((C, nz, na, nd)).astype(np.float32)
    prob = TgvProblem(f, g, (4.0, 1.0), [1.0] * C, dim=3, L=30.0, u0=u0)
    prob.iterate(1, ku_on_last=True)
    want = O.radon_fwd(u0.astype(np.float64), g.ofs.T, nd)
    assert rel(prob.ku.cpu().numpy(), want) <= lines.BAR
    sino = torch.empty((C, nz, na, nd), device="cuda")
    radon(sino, torch.as_tensor(u0, device="cuda"), g)
    assert rel(sino.cpu().numpy(), want) <= lines.BAR


@pytest.mark.parametrize("disc", ["L2", "KL"])
def test_slabs_of_a_gathered_volume_give_its_bits(disc):
    """60 slices of 96 x 96 are gathered; the slabs of 20 alone would go by
    lines.  The gather's own KL prox and gr_prox, which slabs use, round
    differently, so with KL the whole is one slab too."""
    from graptor_amd.projector import RadonGeometry
    from graptor_amd.slabs import SlabSolve
    from graptor_amd.solver import TgvProblem
    C, nz, na = 4, 15, 40
    print(f"slabs of {C} x {nz} {disc}", flush=True)
    g = RadonGeometry((96, 96), angles_deg(-70, 70, na), n_detectors=96)
    assert not g.iterates_by_lines(C * nz) and g.iterates_by_lines(C * nz // 3)
    f = np.random.default_rng(nz).random((C, nz, na, 96)).astype(np.float32)
    kw = dict(coupling="frobenius", discrepancy=disc, L=40.0)
    if disc == "KL":
        whole = SlabSolve(f, g, (4.0, 1.0), [1.0] * C, 1, **kw)
        of_whole = whole.gather
    else:
        whole = TgvProblem(f, g, (4.0, 1.0), [1.0] * C, dim=3, **kw)
        of_whole = lambda name: getattr(whole, name)
    parts = SlabSolve(f, g, (4.0, 1.0), [1.0] * C, 3, **kw)
    whole.iterate(6)
    parts.iterate(6)
    for name in ("u", "v", "lam", "ktl"):
        assert torch.equal(of_whole(name), parts.gather(name)), name


@pytest.mark.parametrize("fuse", [False, True])
def test_part_of_a_stack_follows_the_iteration(fuse):
    """A fused primal step leaves no scratch to the projection, so iterations
    gather; parts of their stack have to as well."""
    from graptor_amd import _lib
    from graptor_amd.projector import RadonGeometry
    from graptor_amd.solver import TgvProblem
    C, N, na = 3, 96, 30
    g = RadonGeometry((N, N), angles_deg(-70, 70, na), n_detectors=N)
    g.set_fusion(fuse)
    assert g.iterates_by_lines(C) != fuse
    rng = np.random.default_rng(7)
    u0 = rng.random((C, 1, N, N)).astype(np.float32)
    f = rng.random((C, 1, na, N)).astype(np.float32)
    prob = TgvProblem(f, g, (4.0, 1.0), [1.0] * C, dim=2, L=30.0, u0=u0)
    prob.iterate(1, ku_on_last=True)
    img = torch.as_tensor(u0[:1, 0].copy(), device="cuda")
    scratch = torch.empty_like(img)
    sino = torch.empty((1, na, N), device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    _lib.check(_lib.load().gr_radon_scratch(g.handle, sino.data_ptr(), img.data_ptr(), 1,
                                            scratch.data_ptr(), C, stream))
    assert torch.equal(sino[0], prob.ku[0, 0])
