"""Iterations of small problems, whose backprojection applies the u half of the
primal step, against the FP32 restatement of the reference kernels: every
dimension and regulariser of that kernel, ragged sizes, several slices."""
import numpy as np
import pytest

from oracle import cref
from oracle import tgv_oracle as O
from tests.helpers import angles_deg, make_problem, rel

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dim,C,nz,N,na,reg,disc", [
    (2, 1, 1, 33, 20, "TGV", "KL"), (2, 3, 1, 65, 31, "TV", "L2"), (3, 1, 2, 30, 18, "TGV", "L2"),
    (3, 2, 5, 67, 260, "TV", "KL"), (2, 2, 1, 130, 40, "TGV", "KL")])
def test_small_iterations(dim, C, nz, N, na, reg, disc):
    from graptor_amd.projector import RadonGeometry
    from graptor_amd.solver import TgvProblem
    print(f"small {dim}D {C} x {nz} x {N} {reg} {disc}", flush=True)
    _, f, ofs = make_problem(5, C, nz, N, na, poisson=50.0)
    f = f.astype(np.float32)
    L = O.normest_power(ofs, N, N, N, iters=40, tol=1e-8)
    g = RadonGeometry((N, N), angles_deg(-70, 70, na), n_detectors=N)
    np.testing.assert_array_equal(g.ofs.T, ofs)
    mu = [1.0, 0.3, 0.2][:C]
    prob = TgvProblem(f, g, (4.0, 1.0), mu, dim=dim, coupling="uncorrelated", discrepancy=disc,
                      regularisation=reg, L=L)
    prob.iterate(20)
    got, ktl = prob.u.cpu().numpy(), prob.ktl.cpu().numpy()
    ref = cref.solve(f, ofs, alpha=(4.0, 1.0), mu=mu, maxiter=20, L=L, coupling="uncorrelated",
                     discrepancy=disc, regularisation=reg, dim=dim)
    # FP32 projections are 1e-6 apart and every iteration adds its own; the
    # solver's bar after N iterations is 1e-3
    assert rel(got, ref["u"]) <= 1e-4
    back = O.radon_adj(prob.lam.cpu().numpy().astype(np.float64), ofs, N, N)
    assert rel(ktl, back) <= 1e-5  # the projector's own bar
