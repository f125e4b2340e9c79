"""Geometries that are never projected by lines are told by one slice: the rule
takes no stack whose single slices it refuses."""
import pytest

from tests.helpers import angles_deg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("N,na,width,lines", [
    (79, 20, 1.0, False), (80, 20, 1.0, True), (80, 266, 1.0, True), (80, 267, 1.0, False),
    (200, 90, 0.9, False), (200, 90, 1.3, False), (200, 90, 1.0, True)])
def test_one_slice_tells(N, na, width, lines):
    from graptor_amd import _lib
    from graptor_amd.projector import RadonGeometry
    g = RadonGeometry((N, N), angles_deg(-75, 75, na), n_detectors=N, detector_width=width)
    assert g.lines == lines
    for S in (1, 2, 3, 4, 5, 8, 64, 300, 3000):
        n = _lib.load().gr_radon_scratch_floats(g.handle, S)
        assert n in (0, S * N * N) and (g.lines or n == 0)
