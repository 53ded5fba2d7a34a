"""Double-precision solves whose BlockPCG column updates run in one launch
for all columns: blocks past the 64 columns of a launch with columns that stop
part way, and few columns of a system large enough that the residual dots are
not fused.  The spectrum is known in closed form; the bounds are those of the
other double-precision solves (eigenvalues 1e-10, residuals 1e-8)."""
import numpy as np
import pytest

import gcge_oracle as O
from gcge_amd import problems as P
from gcge_amd import solver as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,dim,nev,bs,init,most", [(40, 2, 80, 70, 210, 290), (24, 3, 60, 65, 195, 255),
                                                    (65, 3, 4, 4, 12, 16)])
def test_solve(hip, n, dim, nev, bs, init, most):
    prob = P.stencil_problem(n, dim, nev, bs, init, most)
    r = S.solve_problem(prob, mode="fp64", shift=1, rand="device", seed=1, want_vectors=True)
    k = r.nev_conv
    assert k >= nev
    exact = P.analytic_eigenvalues(n, dim, k)
    assert np.max(np.abs(r.eval[:k] - exact) / exact) <= 1e-10
    rr = O.relative_residuals(prob.A, prob.B, r.eval[:k], r.evec[:, :k])
    assert rr.max() <= 1.01e-8
