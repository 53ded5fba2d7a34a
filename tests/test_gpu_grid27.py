"""27-point grid operators: the products that take the neighbours by grid
position against the general sparse kernels of the same matrix, bit for bit,
and against the CPU product where the matrix is uploaded from the host."""
import ctypes as C

import numpy as np
import pytest

import gcge_oracle as O
from gcge_amd import abi, problems as P, solver as S
from gcge_amd.solver import DeviceMatrix, HipTable

pytestmark = pytest.mark.gpu


def ia(*v):
    return (C.c_int * len(v))(*v)


def operator(n, general, fp32=False, seed=3):
    k = np.exp(np.random.default_rng(seed).standard_normal(n ** 3))
    return DeviceMatrix.grid(P.GRID_KINDS["diffusion"], 3, 27, n, k, 1e-8, fp32, general)


def product(table, mat, x, x_off=0, y_off=0):
    n, k = x.shape
    hx = table.create_multivec(k + x_off, mat)
    hy = table.create_multivec(k + y_off, mat)
    table.upload(hx, x, x_off)
    table.slot("MatDotMultiVec")(mat.handle, hx, hy, ia(x_off, y_off), ia(x_off + k, y_off + k),
                                 table.ops)
    y = table.download(hy, y_off, y_off + k, n)
    table.destroy_multivec(hx, k + x_off)
    table.destroy_multivec(hy, k + y_off)
    return y


# lines shorter than a wavefront's 128 points, of exactly 128, cut in chunks,
# odd and even
@pytest.mark.parametrize("n", [4, 5, 16, 31, 64, 65, 127, 128, 129, 130])
def test_product_bits(hip, n):
    table = HipTable()
    grid, gen = operator(n, False), operator(n, True)
    for k, x_off, y_off in ((1, 0, 0), (3, 1, 0)) if n > 100 else ((1, 0, 1), (2, 3, 0), (7, 0, 0)):
        x = np.random.default_rng([n, k]).standard_normal((n ** 3, k))
        assert np.array_equal(product(table, grid, x, x_off, y_off), product(table, gen, x))


@pytest.mark.parametrize("n", [5, 6, 21])
def test_non_finite_values_stay_with_their_neighbours(hip, n):
    table = HipTable()
    grid, gen = operator(n, False), operator(n, True)
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n ** 3, 4))
    for c, v in enumerate((np.nan, np.inf, -np.inf, np.inf)):
        x[rng.integers(0, n ** 3, 3), c] = v
    x[[0, n - 1, n, n * n - 1, n ** 3 - 1], 3] = np.inf
    a, b = product(table, grid, x), product(table, gen, x)
    # the CPU product says which values are infinite or NaN (the general
    # kernels' padding entries, 0 times the row's own value, make NaN of an
    # infinity in a boundary row itself)
    k = np.exp(np.random.default_rng(3).standard_normal(n ** 3))
    with np.errstate(invalid="ignore"):
        ref = O.spmm(P.varcoef27_from(n, k, 1e-8), x)
    fine = np.isfinite(ref)
    assert np.array_equal(np.where(fine, 0.0, a), np.where(fine, 0.0, ref), equal_nan=True)
    assert np.array_equal(a[fine], b[fine])


def test_uploaded_matrices(hip):
    """Recognised from host arrays; a matrix off the pattern by one entry, or
    with one entry's place exchanged, keeps the general kernels' results."""
    table = HipTable()
    n = 9
    A = P.varcoef27_pair(n, 1.0, np.random.default_rng(2))[0]
    x = np.random.default_rng(4).standard_normal((n ** 3, 5))
    ref = O.spmm(A, x)
    assert np.array_equal(product(table, DeviceMatrix(A), x),
                          product(table, DeviceMatrix(A, general=True), x))
    for i, j in ((0, 1), (40, 41), (n ** 3 - 1, n ** 3 - 2)):
        Z = A.tolil()
        Z[i, j] = Z[j, i] = 0.0
        Z = Z.tocsc()
        Z.sort_indices()
        far = A.tolil()
        far[i, (i + 3 * n * n) % n ** 3] = far[(i + 3 * n * n) % n ** 3, i] = 0.5
        far = far.tocsc()
        far.sort_indices()
        for M in (Z, far):
            y, want = product(table, DeviceMatrix(M), x), O.spmm(M, x)
            assert np.max(np.abs(y - want)) <= 1e-13 * np.max(np.abs(want))
    assert np.max(np.abs(product(table, DeviceMatrix(A), x) - ref)) <= 1e-13 * np.max(np.abs(ref))


@pytest.mark.parametrize("n,k", [(5, 3), (16, 8), (21, 9), (33, 17), (50, 4)])
def test_block_pcg_bits(hip, n, k):
    out = []
    for general in (False, True):
        table = HipTable()
        mat = operator(n, general, fp32=True)
        rng = np.random.default_rng([n, k])
        b, x = rng.standard_normal((n ** 3, k)), rng.standard_normal((n ** 3, k))
        hb, hx = table.create_multivec(k, mat), table.create_multivec(k, mat)
        table.upload(hb, b)
        table.upload(hx, x)
        hip.HIPGCG_MultiLinearSolverSetup_BlockPCG32(30, 1e-3, 1e-14, None, 0.0, table.ops)
        abi.slot(table.ops, "MultiLinearSolver")(mat.handle, hb, hx, ia(0, 0), ia(k, k), table.ops)
        out.append(table.download(hx, 0, k, n ** 3))
        table.destroy_multivec(hb, k)
        table.destroy_multivec(hx, k)
        hip.HIPGCG_MultiLinearSolverFree_BlockPCG32(table.ops)
    assert np.array_equal(out[0], out[1])


def recognised(table, mat):
    """Whether products with the operator run by grid position: an infinite
    value at the first point stays infinite there, where the general kernels'
    padding of its short row, 0 times the value, makes NaN of it."""
    x = np.zeros((mat.n, 1))
    x[0] = np.inf
    return bool(np.isinf(product(table, mat, x)[0, 0]))


# three chunks of x-lines, odd and even, and the largest side that is
# recognised: the offsets into a column and into a tile reach furthest
@pytest.mark.parametrize("n", [249, 250, 256])
def test_product_bits_long_lines(hip, n):
    table = HipTable()
    grid, gen = operator(n, False), operator(n, True)
    assert recognised(table, grid) and not recognised(table, gen)
    x = np.random.default_rng(n).standard_normal((n ** 3, 2))
    assert np.array_equal(product(table, grid, x), product(table, gen, x))


# from 66 on a wavefront's 64 rows can lie inside an x-line, away from its ends
@pytest.mark.parametrize("n,k", [(64, 3), (66, 9), (67, 9), (100, 9), (130, 17), (256, 1)])
def test_block_pcg_bits_inside_lines(hip, n, k):
    out = []
    rng = np.random.default_rng([n, k])
    b, x = rng.standard_normal((n ** 3, k)), rng.standard_normal((n ** 3, k))
    for general in (False, True):
        table = HipTable()
        mat = operator(n, general, fp32=True)
        assert recognised(table, mat) == (not general)
        hb, hx = table.create_multivec(k, mat), table.create_multivec(k, mat)
        table.upload(hb, b)
        table.upload(hx, x)
        hip.HIPGCG_MultiLinearSolverSetup_BlockPCG32(9, 1e-3, 1e-14, None, 0.0, table.ops)
        abi.slot(table.ops, "MultiLinearSolver")(mat.handle, hb, hx, ia(0, 0), ia(k, k), table.ops)
        out.append(table.download(hx, 0, k, n ** 3))
        table.destroy_multivec(hb, k)
        table.destroy_multivec(hx, k)
        hip.HIPGCG_MultiLinearSolverFree_BlockPCG32(table.ops)
    assert np.all(np.isfinite(out[0])) and np.array_equal(out[0], out[1])


def test_uploaded_matrices_are_recognised(hip):
    table, n = HipTable(), 9
    A = P.varcoef27_pair(n, 1.0, np.random.default_rng(2))[0]
    assert recognised(table, DeviceMatrix(A))
    assert not recognised(table, DeviceMatrix(A, general=True))


@pytest.mark.parametrize("mode,shift", [("fp64", 1), ("mixed", 0)])
def test_solve_bits(hip, mode, shift):
    """Whole solves by grid position and on the general 32-entry rows."""
    A, B = P.varcoef27_pair(20, 1.0, np.random.default_rng(8))
    bs, ni, nm = P.slepc_block_policy(20)
    prob = P.CCSProblem("27pt_20", A, B, 20, bs, ni, nm)
    fp32 = mode == "mixed"
    r = [S.solve_problem(prob, mode=mode, shift=shift, rand="device", seed=1, want_vectors=True,
                         mats=(DeviceMatrix(A, fp32, general), DeviceMatrix(B, fp32)))
         for general in (False, True)]
    assert r[0].nev_conv >= 20 and r[0].num_iter == r[1].num_iter
    assert np.array_equal(r[0].eval, r[1].eval) and np.array_equal(r[0].evec, r[1].evec)


@pytest.mark.parametrize("n,few", [(32, False), (33, True), (38, True), (39, False)])
def test_few_columns_on_small_grids(hip, n, few):
    """Up to three columns of these sides take the general kernel."""
    table = HipTable()
    grid, gen = operator(n, False), operator(n, True)
    assert recognised(table, grid) == (not few)
    for k in (1, 3, 4, 5):
        x = np.random.default_rng([n, k]).standard_normal((n ** 3, k))
        assert np.array_equal(product(table, grid, x), product(table, gen, x))
