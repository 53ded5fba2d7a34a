"""The three-launch BlockPCG iteration past 65,536 rows and over wide blocks
against the five-launch one, bit for bit: stencil, 27-point and 2D operators,
with columns that stop part way, eager and from graphs."""
import ctypes as C

import numpy as np
import pytest

from gcge_amd import abi, problems as P
from gcge_amd.solver import DeviceMatrix, HipTable

pytestmark = pytest.mark.gpu


def ia(*v):
    return (C.c_int * len(v))(*v)


def matrix(op, n):
    if op == "lap3d":
        return DeviceMatrix.grid(P.GRID_KINDS["laplace"], 3, 7, n, fp32=True)
    dim, pts = (2, 5) if op == "diff2d" else (3, 27)
    k = np.exp(0.5 * np.random.default_rng(n).standard_normal(n ** dim))
    return DeviceMatrix.grid(P.GRID_KINDS["diffusion"], dim, pts, n, k, 1e-8, True)


# rows and columns on both sides of the row-tile limit; 300 columns exceed the
# columns whose sums one stage holds
@pytest.mark.parametrize("op,n,k", [("lap3d", 44, 20), ("lap3d", 60, 8), ("lap3d", 62, 17),
                                    ("diff27", 41, 9), ("diff27", 52, 20), ("diff2d", 260, 9),
                                    ("diff2d", 350, 24), ("diff2d", 100, 300), ("diff2d", 250, 40)])
def test_three_launches_match_five(hip, op, n, k):
    table, mat = HipTable(), matrix(op, n)
    rows = mat.n
    rng = np.random.default_rng([n, k])
    hb, hx = table.create_multivec(k, mat), table.create_multivec(k, mat)
    # columns of very different smoothness stop at different iterations
    b = rng.standard_normal((rows, k))
    b[:, ::3] = np.cumsum(b[:, ::3], axis=0)
    table.upload(hb, b)
    outs = []
    for fused, graphs in ((1, 0), (0, 0), (1, 1)):
        hip.HIPGCG_MultiLinearSolverSetup_BlockPCG32(45, 0.03, 1e-14, None, 0.0, table.ops)
        hip.HIPGCG_BlockPCG32_SetGraphs(table.ops, graphs)
        hip.HIPGCG_BlockPCG32_SetFused(table.ops, fused)
        table.upload(hx, np.zeros((rows, k)))
        abi.slot(table.ops, "MultiLinearSolver")(mat.handle, hb, hx, ia(0, 0), ia(k, k), table.ops)
        outs.append(table.download(hx, 0, k, rows))
    table.destroy_multivec(hb, k)
    table.destroy_multivec(hx, k)
    hip.HIPGCG_MultiLinearSolverFree_BlockPCG32(table.ops)
    assert np.all(np.isfinite(outs[0]))
    assert np.array_equal(outs[0], outs[1]) and np.array_equal(outs[0], outs[2])
