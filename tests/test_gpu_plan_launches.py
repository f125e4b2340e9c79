"""Batch plans whose problems project forward in different ways: by lines and by
the gather in one launch (small plans), longer lines in a launch of their own,
transposition beside the dual step or ahead of the fork.  Every problem gets the
bits that it gets alone, eagerly and from a graph."""
import numpy as np
import pytest

from tests.helpers import angles_deg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# (image side, angles, channels, regularisation, detector width); by lines from 80
# pixels on: up to 4 waves of items an angle (180 pixels) or more
PLANS = {
    "mixed": [(64, 20, 1, "TGV", 1.0), (97, 23, 1, "TGV", 1.0)],
    "mixed, groups of 1, 2 and 4 slices": [
        (33, 11, 1, "TGV", 1.0), (50, 20, 2, "TGV", 1.0), (79, 25, 5, "TGV", 1.0),
        (80, 13, 1, "TGV", 1.0), (95, 30, 2, "TV", 1.0), (129, 31, 3, "TGV", 1.0)],
    "mixed, lines of more waves, wide bins": [
        (60, 20, 1, "TGV", 1.0), (100, 20, 4, "TGV", 1.0), (330, 40, 1, "TGV", 1.0),
        (60, 20, 2, "TGV", 1.7)],
    "lines of more waves and gather": [(60, 20, 1, "TGV", 1.0), (260, 40, 2, "TGV", 1.0)],
    "lines, one slice": [(90, 20, 1, "TGV", 1.0), (120, 17, 1, "TGV", 1.0)],
    "lines, groups of 2 and 4": [(90, 20, 2, "TGV", 1.0), (120, 17, 4, "TGV", 1.0)],
    "six channels": [(85, 17, 6, "TGV", 1.0), (60, 20, 1, "TGV", 1.0)],
    "nine channels": [(85, 17, 9, "TGV", 1.0), (60, 20, 1, "TGV", 1.0)],
    # more than 2^20 voxel-channels: projections beside the stencil steps
    "overlapped": [(64, 20, 1, "TGV", 1.0), (97, 23, 2, "TGV", 1.0), (560, 60, 4, "TGV", 1.0)],
}


def _problem(i, N, na, C, reg, width):
    from graptor_amd.projector import RadonGeometry
    from graptor_amd.solver import TgvProblem
    g = RadonGeometry((N, N), angles_deg(-80, 80, na), n_detectors=N, detector_width=width)
    assert g.iterates_by_lines(C) == (N >= 80 and width == 1.0)
    rng = np.random.default_rng(10 + i)
    f = rng.random((C, 1, na, N)).astype(np.float32)
    u0 = rng.random((C, 1, N, N)).astype(np.float32)
    return TgvProblem(f, g, (4.0, 1.0), [1.0] * C, dim=2, regularisation=reg, L=float(N), u0=u0)


@pytest.mark.parametrize("name", PLANS)
def test_plan_gives_the_bits_of_each_problem(name):
    from graptor_amd.batch import BatchPlan
    print(name, flush=True)
    specs = PLANS[name]
    alone, eager, graph = ([_problem(i, *s) for i, s in enumerate(specs)] for _ in range(3))
    for p in alone:
        p.iterate(6, ku_on_last=True)
    BatchPlan(eager).iterate(6, ku_on_last=True)
    plan = BatchPlan(graph)
    for _ in range(3):  # one capture, replayed with other work in between
        plan.iterate_graph(2, 2)
        torch.cuda.synchronize()
        torch.ones(1000, device="cuda").sum().item()
    for i, (a, e, g) in enumerate(zip(alone, eager, graph)):
        assert torch.equal(a.ku, e.ku), specs[i]
        for field in ("u", "ubar", "lam", "ktl", "v"):
            assert torch.equal(getattr(a, field), getattr(e, field)), (specs[i], field)
            assert torch.equal(getattr(a, field), getattr(g, field)), (specs[i], field)
