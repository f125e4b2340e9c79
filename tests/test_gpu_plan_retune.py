"""A plan whose retune failed has no work lists: it refuses to iterate, and goes on
where it was once a retune succeeds."""
import numpy as np
import pytest

from tests.helpers import angles_deg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _problem():
    from graptor_amd.projector import RadonGeometry
    from graptor_amd.solver import TgvProblem
    g = RadonGeometry((64, 64), angles_deg(-70, 70, 15), n_detectors=64)
    f = np.random.default_rng(1).random((3, 1, 15, 64)).astype(np.float32)
    return TgvProblem(f, g, (4.0, 1.0), [1.0] * 3, dim=2, L=40.0)


def test_failed_retune():
    from graptor_amd.batch import BatchPlan
    prob, want = _problem(), _problem()
    want.iterate(6)
    plan = BatchPlan([prob])
    plan.iterate(2)
    prob.geometry.set_tuning(fwd_band=256)  # 256 lines of 64 pixels, four slices: 270 KB
    for _ in range(2):
        with pytest.raises(ValueError, match="too large"):
            plan.retune()
        for call in (lambda: plan.iterate(1), lambda: plan.iterate_graph(2, 2),
                     lambda: plan.profile(1)):
            with pytest.raises(ValueError, match="retune failed"):
                call()
    prob.geometry.set_tuning(fwd_band=16)
    plan.retune()
    plan.iterate(2)
    plan.iterate_graph(2, 2)
    assert prob.iterations == 6
    assert torch.equal(prob.u, want.u) and torch.equal(prob.lam, want.lam)
