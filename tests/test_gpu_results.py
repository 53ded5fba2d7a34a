"""Inner products whose values are polled in pinned memory: each call returns
its own values (small whole numbers, whose sums are exact in any order), call
after call into the same buffer, with symmetric blocks and blocks that are
copied back in between, and with results that take longer than the polling;
NaN inputs, among them the pattern that marks a value as awaited, give NaN."""
import ctypes as C

import numpy as np
import pytest

from gcge_amd import abi, problems as P
from gcge_amd.solver import DeviceMatrix, HipTable

pytestmark = pytest.mark.gpu


def inner(table, kind, hx, hy, m, n):
    ip = np.full((m, n), 7.0, order="F")
    table.slot("MultiVecInnerProd")(kind, hx, hy, 0, (C.c_int * 2)(0, 0), (C.c_int * 2)(m, n),
                                    ip.ctypes.data_as(abi.c_dbl_p), 1 if kind == b"D" else m,
                                    table.ops)
    return ip.T.ravel()[:n].copy() if kind == b"D" else ip


@pytest.mark.parametrize("rows", [1, 300, 20011, 2000003])
def test_each_call_its_own(hip, rows):
    rng = np.random.default_rng(rows)
    k = 66 if rows < 100000 else 12
    table, mat = HipTable(), DeviceMatrix(P.diagonal_ccs(np.ones(rows)))
    hx, hy = table.create_multivec(k, mat), table.create_multivec(k, mat)
    for step in range(3):
        x = rng.integers(-3, 4, (rows, k)).astype(float)
        y = rng.integers(-3, 4, (rows, k)).astype(float)
        table.upload(hx, x)
        table.upload(hy, y)
        xy, yy = x.T @ y, y.T @ y
        for m, n in ((1, 1), (k, 1), (3, 9), (k, k), (10, 12), (1, 1)):
            assert np.array_equal(inner(table, b"N", hx, hy, m, n), xy[:m, :n])
            assert np.array_equal(inner(table, b"S", hy, hy, n, n), yy[:n, :n])
            assert np.array_equal(inner(table, b"D", hx, hy, n, n), np.diag(xy)[:n])
    table.destroy_multivec(hx, k)
    table.destroy_multivec(hy, k)


@pytest.mark.parametrize("bits", [0x7FF8000000000000, 0x7FF4A5A5A5A5A5A5])
def test_nan(hip, bits):
    rows, k = 777, 12
    x = np.ones((rows, k))
    x[5, 2] = np.array([bits], dtype=np.uint64).view(float)[0]
    table, mat = HipTable(), DeviceMatrix(P.diagonal_ccs(np.ones(rows)))
    h = table.create_multivec(k, mat)
    table.upload(h, x)
    want = np.full((k, k), float(rows))
    want[2, :] = want[:, 2] = np.nan
    for n in (1, k):
        assert np.array_equal(inner(table, b"N", h, h, k, n), want[:, :n], equal_nan=True)
    assert np.array_equal(inner(table, b"D", h, h, k, k), np.diag(want), equal_nan=True)
    table.destroy_multivec(h, k)
