"""MultiVecLinearComb at the edges of its kernel's tiles: row pairs with one
row past the end, 16-column tiles in one to several column tiles, chunks of 16
source columns, every beta mode, against numpy.

Each value is a chain of at most m multiply-adds (padding adds zeros) and the
product with beta, so its error is below m + 2 units of roundoff of
|x| |c| + |y beta|."""
import ctypes as C

import numpy as np
import pytest

from gcge_amd import abi, problems as P
from gcge_amd.solver import DeviceMatrix, HipTable

pytestmark = pytest.mark.gpu


def ia(*v):
    return (C.c_int * len(v))(*v)


def check(table, mat, rows, m, n, mode, x_off=0, y_off=0):
    rng = np.random.default_rng([rows, m, n, mode])
    x, y = rng.standard_normal((rows, m)), rng.standard_normal((rows, n))
    c = np.asfortranarray(rng.standard_normal((m + 2, n)))
    beta = {0: None, 1: np.array([-0.75]), 2: rng.standard_normal(n)}[mode]
    hx, hy = table.create_multivec(m + x_off, mat), table.create_multivec(n + y_off, mat)
    table.upload(hx, x, x_off)
    table.upload(hy, y, y_off)
    table.slot("MultiVecLinearComb")(
        hx, hy, 0, ia(x_off, y_off), ia(x_off + m, y_off + n), c.ctypes.data_as(abi.c_dbl_p), m + 2,
        beta.ctypes.data_as(abi.c_dbl_p) if mode else None, 1 if mode == 2 else 0, table.ops)
    got = table.download(hy, y_off, y_off + n, rows)
    table.destroy_multivec(hx, m + x_off)
    table.destroy_multivec(hy, n + y_off)
    b = 0.0 if mode == 0 else beta
    want = x @ c[:m] + y * b
    bound = (m + 2) * np.finfo(float).eps * (np.abs(x) @ np.abs(c[:m]) + np.abs(y * b))
    assert np.all(np.abs(got - want) <= bound), (rows, m, n, mode)


@pytest.mark.parametrize("rows", [1, 2, 3, 63, 64, 65, 127, 128, 129, 255, 257, 1001])
def test_row_edges(hip, rows):
    table, mat = HipTable(), DeviceMatrix(P.diagonal_ccs(np.ones(rows)))
    for m, n in ((1, 1), (4, 17), (5, 48), (16, 16), (17, 33), (33, 130)):
        for mode in (0, 1, 2):
            check(table, mat, rows, m, n, mode, x_off=1, y_off=m % 2)


@pytest.mark.parametrize("n", [15, 16, 17, 48, 64, 65, 96, 112, 113, 128, 129, 144, 145, 160, 290])
def test_column_tiles(hip, n):
    rows = 777
    table, mat = HipTable(), DeviceMatrix(P.diagonal_ccs(np.ones(rows)))
    for m in (1, 15, 31, 32, 50):
        for mode in (0, 1, 2):
            check(table, mat, rows, m, n, mode)


@pytest.mark.parametrize("n", [9, 30, 40, 60])
def test_tall_tiles(hip, n):
    """Enough rows for 64 per wave (512 workgroups of 256), odd."""
    rows = 131073
    table, mat = HipTable(), DeviceMatrix(P.diagonal_ccs(np.ones(rows)))
    for m, mode in ((3, 0), (20, 1), (17, 2)):
        check(table, mat, rows, m, n, mode)


def test_offsets_past_32_bits(hip):
    """2^27 rows: three columns reach past the 32-bit offsets of a load."""
    rows = 1 << 27
    table = HipTable()
    mat = DeviceMatrix.grid(P.GRID_KINDS["diagonal"], 1, 0, rows, np.ones(rows))
    hx, hy = table.create_multivec(2, mat), table.create_multivec(1, mat)
    hip.gcge_hip_set_random_mode(abi.GCGE_HIP_RAND_DEVICE, 5)
    table.slot("MultiVecSetRandomValue")(hx, 0, 2, table.ops)
    hip.gcge_hip_set_random_mode(abi.GCGE_HIP_RAND_LIBC, 0)
    c = np.array([1.25, -0.5])
    table.slot("MultiVecLinearComb")(hx, hy, 0, ia(0, 0), ia(2, 1), c.ctypes.data_as(abi.c_dbl_p), 2,
                                     None, 0, table.ops)
    want = table.download(hx, 0, 1, rows)[:, 0] * c[0]
    want += table.download(hx, 1, 2, rows)[:, 0] * c[1]
    got = table.download(hy, 0, 1, rows)[:, 0]
    table.destroy_multivec(hx, 2)
    table.destroy_multivec(hy, 1)
    got -= want
    # two products and a sum of values below 1.25
    assert max(got.max(), -got.min()) <= 3 * np.finfo(float).eps * 1.75


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_offsets_past_32_bits_with_beta(hip, mode):
    """More than 2^27 rows, an odd number, in two 16-column tiles, against the
    same sums column by column (MultiVecAxpby).  Values lie in [0, 1), so each
    side is within m + 2 units of roundoff of the sum of |c| and |beta|, and
    one wrong value in 134 M stands out of the norm of all differences."""
    rows, m, n = (1 << 27) + 1, 5, 18
    table = HipTable()
    axpby = table.slot("MultiVecAxpby")
    mat = DeviceMatrix.grid(P.GRID_KINDS["diagonal"], 1, 0, rows, np.ones(rows))
    hx, hy, hz = (table.create_multivec(k, mat) for k in (m, n, n))
    hip.gcge_hip_set_random_mode(abi.GCGE_HIP_RAND_DEVICE, 5)
    table.slot("MultiVecSetRandomValue")(hx, 0, m, table.ops)
    table.slot("MultiVecSetRandomValue")(hy, 0, n, table.ops)
    hip.gcge_hip_set_random_mode(abi.GCGE_HIP_RAND_LIBC, 0)
    rng = np.random.default_rng(mode)
    c = np.asfortranarray(rng.uniform(-1, 1, (m, n)))
    beta = {0: None, 1: np.array([-0.75]), 2: rng.uniform(-1, 1, n)}[mode]
    b = np.broadcast_to(0.0 if beta is None else beta, n)
    axpby(1.0, hy, 0.0, hz, ia(0, 0), ia(n, n), table.ops)
    for j in range(n):
        axpby(0.0, None, b[j], hz, ia(j, j), ia(j + 1, j + 1), table.ops)
        for k in range(m):
            axpby(c[k, j], hx, 1.0, hz, ia(k, j), ia(k + 1, j + 1), table.ops)
    table.slot("MultiVecLinearComb")(
        hx, hy, 0, ia(0, 0), ia(m, n), c.ctypes.data_as(abi.c_dbl_p), m,
        beta.ctypes.data_as(abi.c_dbl_p) if mode else None, 1 if mode == 2 else 0, table.ops)
    axpby(-1.0, hz, 1.0, hy, ia(0, 0), ia(n, n), table.ops)
    d = np.empty(n)
    table.slot("MultiVecInnerProd")(b"D", hy, hy, 0, ia(0, 0), ia(n, n),
                                    d.ctypes.data_as(abi.c_dbl_p), 1, table.ops)
    for h, k in ((hx, m), (hy, n), (hz, n)):
        table.destroy_multivec(h, k)
    each = 2 * (m + 2) * np.finfo(float).eps * (np.abs(c).sum(axis=0) + np.abs(b))
    assert np.all(np.sqrt(d) <= np.sqrt(rows) * each)


# both sides of each limit of the library GEMM: 448 Ki rows, 100 source
# columns, destination columns whose sixteens are a multiple of 8 (113-128,
# 241-256), no beta per column
@pytest.mark.parametrize("rows,m,n,mode", [(458752, 100, 113, 0), (458753, 101, 128, 1),
                                           (458752, 100, 128, 2), (458751, 100, 128, 1),
                                           (458752, 99, 128, 0), (458752, 100, 112, 1),
                                           (458752, 100, 129, 1), (458752, 100, 241, 1)])
def test_library_limits(hip, rows, m, n, mode):
    check(HipTable(), DeviceMatrix(P.diagonal_ccs(np.ones(rows))), rows, m, n, mode)


def launches(hip, kind):
    n, ms, b, f = C.c_int64(), C.c_double(), C.c_double(), C.c_double()
    hip.gcge_hip_profile_read(kind, C.byref(n), C.byref(ms), C.byref(b), C.byref(f))
    return n.value


# from 512,000 rows on the library also takes widths for which the kernel's
# tiles hold as much padding (225-240, 353-368), and with beta and few source
# columns an eighth less (112, 300); the alignment of the columns' starts, the
# source columns and the rows on both sides of their limits
@pytest.mark.parametrize("rows,m,n,mode,library", [
    (512000, 100, 240, 0, True), (511999, 100, 240, 0, False), (512004, 100, 240, 0, False),
    (512004, 255, 240, 0, False), (512004, 256, 240, 0, True), (512004, 100, 240, 1, True), (512001, 230, 240, 1, False), (512008, 230, 225, 1, True),
    (512000, 230, 224, 1, False), (512000, 223, 224, 1, True), (512000, 224, 112, 1, False),
    (512000, 100, 112, 1, True), (512000, 100, 112, 0, False), (512000, 99, 112, 1, False),
    (512000, 120, 300, 1, True), (512000, 120, 300, 0, False), (512000, 120, 355, 0, True),
    (512000, 100, 192, 1, False), (511984, 100, 225, 1, False)])
def test_library_widths(hip, rows, m, n, mode, library):
    """Which of the two runs, and its values against the kernel with the same
    beta per column (never the library).  Values lie in [0, 1): each side is
    within m + 2 units of roundoff of the sum of |c| and |beta|."""
    table = HipTable()
    mat = DeviceMatrix.grid(P.GRID_KINDS["diagonal"], 1, 0, rows, np.ones(rows))
    hx, hy, hz = (table.create_multivec(k, mat) for k in (m, n, n))
    hip.gcge_hip_set_random_mode(abi.GCGE_HIP_RAND_DEVICE, 7)
    table.slot("MultiVecSetRandomValue")(hx, 0, m, table.ops)
    table.slot("MultiVecSetRandomValue")(hy, 0, n, table.ops)
    hip.gcge_hip_set_random_mode(abi.GCGE_HIP_RAND_LIBC, 0)
    axpby, comb = table.slot("MultiVecAxpby"), table.slot("MultiVecLinearComb")
    axpby(1.0, hy, 0.0, hz, ia(0, 0), ia(n, n), table.ops)
    c = np.asfortranarray(np.random.default_rng(n).uniform(-1, 1, (m, n)))
    one, each = np.array([0.625]), np.full(n, 0.625 if mode else 0.0)
    hip.gcge_hip_profile_enable(1)
    hip.gcge_hip_profile_reset()
    comb(hx, hy, 0, ia(0, 0), ia(m, n), c.ctypes.data_as(abi.c_dbl_p), m,
         one.ctypes.data_as(abi.c_dbl_p) if mode else None, 0, table.ops)
    gemm, own = launches(hip, 6), launches(hip, 3)
    hip.gcge_hip_profile_enable(0)
    assert (gemm, own) == ((1, 0) if library else (0, 1))
    comb(hx, hz, 0, ia(0, 0), ia(m, n), c.ctypes.data_as(abi.c_dbl_p), m,
         each.ctypes.data_as(abi.c_dbl_p), 1, table.ops)
    axpby(-1.0, hz, 1.0, hy, ia(0, 0), ia(n, n), table.ops)
    d = np.empty(n)
    table.slot("MultiVecInnerProd")(b"D", hy, hy, 0, ia(0, 0), ia(n, n),
                                    d.ctypes.data_as(abi.c_dbl_p), 1, table.ops)
    for h, k in ((hx, m), (hy, n), (hz, n)):
        table.destroy_multivec(h, k)
    bound = 2 * (m + 2) * np.finfo(float).eps * (np.abs(c).sum(axis=0) + each)
    assert np.all(np.sqrt(d) <= np.sqrt(rows) * bound)


@pytest.mark.parametrize("rows", [130, 131073])
@pytest.mark.parametrize("n", [16, 17, 32, 33])
def test_one_chunk_of_coefficients(hip, rows, n):
    """At most 16 source columns into at most 32, and one more of each."""
    table, mat = HipTable(), DeviceMatrix(P.diagonal_ccs(np.ones(rows)))
    for m, mode in ((15, 1), (16, 0), (16, 2), (17, 1)):
        check(table, mat, rows, m, n, mode)
