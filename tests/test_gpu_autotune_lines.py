"""The autotuner sets no forward band where there is none: problems that project
by lines keep the automatic one, whatever is tuned beside them."""
import numpy as np
import pytest

from tests.helpers import angles_deg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _problem(N, na):
    from graptor_amd.projector import RadonGeometry
    from graptor_amd.solver import TgvProblem
    g = RadonGeometry((N, N), angles_deg(-70, 70, na), n_detectors=N)
    f = np.random.default_rng(N).random((1, 1, na, N)).astype(np.float32)
    return TgvProblem(f, g, (4.0, 1.0), [1.0], dim=2, coupling="uncorrelated", L=float(N))


@pytest.mark.parametrize("beside", [False, True])
def test_lines_have_no_band(tmp_path, beside):
    from graptor_amd.autotune import autotune
    lines, gather = _problem(100, 25), _problem(40, 20)
    assert lines.geometry.iterates_by_lines(1) and not gather.geometry.iterates_by_lines(1)
    lines.geometry.set_fusion(True)  # the fused primal step gathers
    assert not lines.geometry.iterates_by_lines(1)
    lines.geometry.set_fusion(False)
    probs = [lines, gather] if beside else [lines]
    cache = str(tmp_path / "tuned.json")
    for _ in range(2):  # the second time from the cache
        res = autotune(probs, iters=1, cache=cache)
        assert lines.geometry.get_tuning() == (0, res["adj_tile_y"])
        assert (res["fwd_band"] > 0) == beside
        if beside:
            assert gather.geometry.get_tuning() == (res["fwd_band"], res["adj_tile_y"])
