"""The tables of the projection by lines are there once a geometry is: for calls
from several threads and streams at once, and inside a capture that makes the
first call."""
import threading

import numpy as np
import pytest

from oracle import tgv_oracle as O
from tests.helpers import angles_deg, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

N, NA = 200, 60


def _geometry():
    from graptor_amd.projector import RadonGeometry
    g = RadonGeometry((N, N), angles_deg(-70, 70, NA), n_detectors=N)
    assert g.iterates_by_lines(1)
    return g


def test_first_calls_from_several_threads_and_streams():
    from graptor_amd.projector import radon
    T = 8
    img = torch.rand((1, N, N), device="cuda")
    sino = torch.empty((T, 1, NA, N), device="cuda")
    torch.cuda.synchronize()
    g = _geometry()
    start = threading.Barrier(T)

    def work(t):
        stream = torch.cuda.Stream()
        start.wait()
        with torch.cuda.stream(stream):
            radon(sino[t], img, g)
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(t,)) for t in range(T)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    want = O.radon_fwd(img.double().cpu().numpy(), g.ofs.T.copy(), N)
    assert rel(sino[0].cpu().numpy(), want) <= 1e-5  # the projector's own bar
    for t in range(1, T):
        assert torch.equal(sino[t], sino[0]), t


def test_first_call_inside_a_capture():
    from graptor_amd import _lib
    lib = _lib.load()
    rng = np.random.default_rng(3)
    img, other = (torch.as_tensor(rng.random((1, N, N)).astype(np.float32), device="cuda")
                  for _ in range(2))
    sino, want = (torch.empty((1, NA, N), device="cuda") for _ in range(2))
    scratch = torch.empty_like(img)
    g = _geometry()

    def call(out):
        _lib.check(lib.gr_radon_scratch(g.handle, out.data_ptr(), img.data_ptr(), 1,
                                        scratch.data_ptr(), 0,
                                        torch.cuda.current_stream().cuda_stream))

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(sino)
    for k in range(4):
        if k % 2:
            img.copy_(other)
        img.mul_(1.5)
        sino.zero_()
        graph.replay()
        torch.cuda.synchronize()
        call(want)
        assert torch.equal(sino, want), k
