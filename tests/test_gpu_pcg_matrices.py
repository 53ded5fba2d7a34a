"""The single-precision BlockPCG's captured iterations belong to the matrix
they were captured with: matrices of the same size, created one after the
other (each destroyed before the next, so that their device arrays can lie at
the same addresses) and solved with on one table without another setup, give
the results of a table of their own, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from gcge_amd import abi, problems as P
from gcge_amd.solver import DeviceMatrix, HipTable

pytestmark = pytest.mark.gpu

N, COLS = 16, 5


def ia(*v):
    return (C.c_int * len(v))(*v)


def with_far_entry(A, i):
    """A with one more pair of entries, between points three planes apart."""
    j = i + 3 * N * N
    M = A.tolil()
    M[i, j] = M[j, i] = 0.5
    M[i, i] += 1.0
    M[j, j] += 1.0
    M = M.tocsc()
    M.sort_indices()
    return M


def with_diagonal(A, i):
    M = A.copy().tolil()
    M[i, i] += 3.0
    M = M.tocsc()
    M.sort_indices()
    return M


def grid27():
    """27-point operators (by grid position) and ones off that pattern."""
    A, B = (P.varcoef27_pair(N, 1.0, np.random.default_rng(s))[0] for s in (1, 2))
    return [A, B, with_far_entry(A, 5), A, with_far_entry(B, 6), B]


def stencil7():
    """Constant coefficients (matrix-free), other constants, one value off."""
    A, B = P.stencil_pair(N, 3)
    return [A, B, with_diagonal(A, 9), A, with_diagonal(B, 2000), 2.0 * A]


@pytest.mark.parametrize("matrices", [grid27, stencil7])
def test_each_matrix_its_own_iterations(hip, matrices):
    mats, rows = matrices(), N ** 3
    b = np.random.default_rng(3).standard_normal((rows, COLS))

    def results(table, mats):
        size = DeviceMatrix(P.diagonal_ccs(np.ones(rows)))
        hb, hx = table.create_multivec(COLS, size), table.create_multivec(COLS, size)
        table.upload(hb, b)
        # rate 0: no column stops, every call replays whole groups
        hip.HIPGCG_MultiLinearSolverSetup_BlockPCG32(30, 0.0, 0.0, None, 0.0, table.ops)
        out = []
        for A in mats:
            mat = DeviceMatrix(A, fp32=True)
            table.upload(hx, np.zeros_like(b))
            abi.slot(table.ops, "MultiLinearSolver")(mat.handle, hb, hx, ia(0, 0),
                                                     ia(COLS, COLS), table.ops)
            out.append(table.download(hx, 0, COLS, rows))
            mat.free()
        table.destroy_multivec(hb, COLS)
        table.destroy_multivec(hx, COLS)
        hip.HIPGCG_MultiLinearSolverFree_BlockPCG32(table.ops)
        return out

    got = results(HipTable(), mats)
    for k, A in enumerate(mats):
        want, = results(HipTable(), [A])
        assert np.all(np.isfinite(want))
        assert np.array_equal(got[k], want), k
