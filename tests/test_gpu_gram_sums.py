"""The sums of the Gram kernels' partial tiles over their row chunks, at the
chunk counts where the summation kernel's rounds of 128 chunks begin and end,
against numpy.

A thin Gram has one row chunk per 1,024 rows up to 512 chunks.  Each entry is
a chain of at most 4 row products per thread and chunk, 8 levels of sums in
the workgroup and the sum over at most 512 chunks, each step rounding once,
so its error is below 530 units of roundoff of sum |x| |y|.
"""
import ctypes as C

import numpy as np
import pytest

from gcge_amd import abi, problems as P
from gcge_amd.solver import DeviceMatrix, HipTable

pytestmark = pytest.mark.gpu


def check(rows, m, n):
    rng = np.random.default_rng([rows, m, n])
    table = HipTable()
    mat = DeviceMatrix(P.diagonal_ccs(np.ones(rows)))
    x, y = rng.standard_normal((rows, m)), rng.standard_normal((rows, n))
    hx, hy = table.create_multivec(m, mat), table.create_multivec(n, mat)
    table.upload(hx, x)
    table.upload(hy, y)
    ip = np.full((m + 2, n), 7.0, order="F")  # rows past m stay as they are
    table.slot("MultiVecInnerProd")(b"N", hx, hy, 0, (C.c_int * 2)(0, 0), (C.c_int * 2)(m, n),
                                    ip.ctypes.data_as(abi.c_dbl_p), m + 2, table.ops)
    table.destroy_multivec(hx, m)
    table.destroy_multivec(hy, n)
    bound = 530 * np.finfo(float).eps * (np.abs(x).T @ np.abs(y))
    assert np.all(np.abs(ip[:m] - x.T @ y) <= bound)
    assert np.all(ip[m:] == 7.0)


@pytest.mark.parametrize("chunks", [1, 2, 16, 127, 128, 129, 256, 511])
@pytest.mark.parametrize("m,n", [(1, 1), (40, 1), (3, 9)])
def test_chunk_sums(hip, chunks, m, n):
    check(1024 * chunks - (chunks * 37) % 500, m, n)


@pytest.mark.parametrize("rows", [1, 63, 300, 1025, 4099])
@pytest.mark.parametrize("m,n", [(1, 2), (7, 3), (8, 4), (9, 5), (17, 8), (65, 1), (2, 33)])
def test_thin_tiles(hip, rows, m, n):
    """Column tiles of 8 with remainders on both sides, thin on either side."""
    check(rows, m, n)


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 33, 129, 1000, 5001])
def test_narrow_tiles(hip, rows):
    """A side of 9 to 64 columns against one of up to several tiles, either
    way round: every width of tile and stages of 16 rows with remainders.
    (At these row counts an entry's sum is a chain of at most 512 rows per
    wave and chunk, 4 waves and the chunks: below 530 roundings.)"""
    for m, n in ((9, 9), (16, 10), (17, 16), (33, 17), (64, 33), (65, 64), (100, 40), (113, 48),
                 (129, 20), (200, 60), (12, 70), (40, 150), (64, 65)):
        check(rows, m, n)
