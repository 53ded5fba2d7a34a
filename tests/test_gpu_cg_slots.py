"""The double-precision BlockPCG calls the slots that a table has: one whose
MultiVecAxpby or MultiVecLocalInnerProd is the caller's own gets its column
updates and residual products through it, call by call, and (the caller's
forwarding to the library's) the same bits as the updates of all columns in
one launch."""
import ctypes as C

import numpy as np
import pytest

from gcge_amd import abi, problems as P
from gcge_amd import solver as S

pytestmark = pytest.mark.gpu


def table_with(name, seen):
    """HipTable whose slot `name` calls seen(*arguments) and the library's."""

    class Table(S.HipTable):
        def __init__(self):
            super().__init__()
            inner = self.slot(name)

            def own(*args):
                seen(*args)
                inner(*args)

            self._own = abi.SIG[name](own)
            setattr(self.ops.contents, name, C.cast(self._own, C.c_void_p).value)

    return Table


def solve(prob):
    return S.solve_problem(prob, mode="fp64", shift=0, rand="device", seed=1, want_vectors=True)


# few columns; several launches' worth of them (more than 64 in a block); a
# system whose residual products are not fused with the update
@pytest.mark.parametrize("n,dim,nev,bs,init,most",
                         [(24, 2, 6, 4, 12, 18), (40, 2, 80, 70, 210, 290), (65, 3, 4, 4, 12, 16)])
def test_own_slots_are_called(hip, monkeypatch, n, dim, nev, bs, init, most):
    prob = P.stencil_problem(n, dim, nev, bs, init, most)
    count = {"update": 0, "residual": 0, "product": 0}

    def axpby(alpha, x, beta, y, *rest):
        # x += alpha p and r -= alpha w, the only ones of this form without a shift
        count["update"] += x is not None and beta == 1.0 and abs(alpha) != 1.0

    def dot(kind, x, y, *rest):
        count["residual"] += kind == b"D" and x == y

    def product(*args):
        count["product"] += 1

    base = solve(prob)
    for name, seen, what in (("MultiVecAxpby", axpby, "update"),
                             ("MultiVecLocalInnerProd", dot, "residual"),
                             ("MatDotMultiVec", product, "product")):
        with monkeypatch.context() as m:
            m.setattr(S, "HipTable", table_with(name, seen))
            r = solve(prob)
        assert count[what] > 0, name
        # (an own product also keeps the 3D operators' fused residual out)
        if name != "MatDotMultiVec" or dim == 2:
            assert r.num_iter == base.num_iter
            assert np.array_equal(r.eval, base.eval) and np.array_equal(r.evec, base.evec), name
