"""The tables of the projection by lines are built by the first call that needs
them: not with the geometry, once for all threads, never inside a capture."""
import threading

import numpy as np
import pytest

from tests.helpers import angles_deg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def test_geometries_without_a_projection_stay_small():
    """1000 angles of 512 x 512: 13 MB of tables, 0.1 MB of everything else."""
    from graptor_amd.projector import RadonGeometry, radon, radon_ad
    N, na = 512, 1000
    img = torch.rand((1, N, N), device="cuda")
    sino, tmp = torch.empty((1, na, N), device="cuda"), torch.empty_like(img)
    del tmp  # the scratch of the projection comes from torch's cache
    # the kernels' code is loaded at their first launches
    few = RadonGeometry((N, N), angles_deg(0, 180, 5), n_detectors=N)
    radon(sino[:, :5].contiguous(), img, few)
    radon_ad(img, sino[:, :5].zero_().contiguous(), few)
    before = _free()
    g = RadonGeometry((N, N), angles_deg(0, 180, na), n_detectors=N)
    radon_ad(img, sino.zero_(), g)
    assert before - _free() < 6 << 20
    radon(sino, img, g)
    assert before - _free() > 10 << 20


def test_threads_share_the_tables():
    from graptor_amd.projector import RadonGeometry, radon
    N, na, T = 200, 60, 8
    img = torch.rand((1, N, N), device="cuda")
    sino = torch.empty((T + 1, 1, na, N), device="cuda")
    g = RadonGeometry((N, N), angles_deg(-70, 70, na), n_detectors=N)
    start = threading.Barrier(T)

    def work(t):
        start.wait()
        radon(sino[t], img, g)

    threads = [threading.Thread(target=work, args=(t,)) for t in range(T)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    radon(sino[T], img, g)
    torch.cuda.synchronize()
    assert float(sino[T].abs().sum()) > 0
    for t in range(T):
        assert torch.equal(sino[t], sino[T]), t


@pytest.mark.parametrize("prepared", [False, True])
def test_capture_without_and_with_tables(prepared):
    """Without tables a captured call gathers; with them it goes by lines."""
    from graptor_amd import _lib
    from graptor_amd.projector import RadonGeometry
    lib = _lib.load()
    N, na = 200, 60
    rng = np.random.default_rng(3)
    img, other = (torch.as_tensor(rng.random((1, N, N)).astype(np.float32), device="cuda")
                  for _ in range(2))
    sino, want = (torch.empty((1, na, N), device="cuda") for _ in range(2))
    scratch = torch.empty_like(img)
    g = RadonGeometry((N, N), angles_deg(-70, 70, na), n_detectors=N)
    if prepared:
        g.prepare(1)

    def call(out, src, lines):
        st = torch.cuda.current_stream().cuda_stream
        if lines:
            _lib.check(lib.gr_radon_scratch(g.handle, out.data_ptr(), src.data_ptr(), 1,
                                            scratch.data_ptr(), 0, st))
        else:
            _lib.check(lib.gr_radon(g.handle, out.data_ptr(), src.data_ptr(), 1, st))

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(sino, img, True)
    for k in range(4):
        img.copy_(other if k % 2 else img)
        img.mul_(1.5)
        sino.zero_()
        graph.replay()
        torch.cuda.synchronize()
        call(want, img, prepared)  # by lines only once the tables are there
        assert torch.equal(sino, want), k
