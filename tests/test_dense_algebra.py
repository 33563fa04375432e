"""The EnKF analysis' dense algebra (adamantine_amd/csrc/adm_dense.hpp),
compiled alone for the host: both of its bodies against numpy."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

SRC = os.path.join(os.path.dirname(__file__), "cxx", "dense_algebra.cpp")
EPS = np.finfo(np.float64).eps


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("dense") / "dense_algebra.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-fPIC",
                    "-shared", "-o", out, SRC], check=True)
    return C.CDLL(out)


@pytest.fixture(params=[0, 1], ids=["plain", "avx2"])
def body(request, lib):
    if not lib.has_body(request.param):
        pytest.skip("the processor has no AVX2")
    return request.param


def ptr(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


def solve(lib, body, A, B):
    A, X = np.array(A, float, order="C"), np.array(B, float, order="C")
    return lib.lu(body, A.shape[0], ptr(A), X.shape[1], ptr(X)), X


@pytest.mark.parametrize("m,nrhs", [(1, 1), (2, 3), (7, 5), (33, 16),
                                    (64, 64), (120, 9)])
def test_lu(lib, body, m, nrhs):
    """A matrix without structure, whose first rows have to be swapped."""
    rng = np.random.RandomState(m)
    A = rng.uniform(-1.0, 1.0, (m, m))
    if m > 1:
        A[0, 0] = 0.0
        A[1, 0] = 1e-8
    B = rng.uniform(-1.0, 1.0, (m, nrhs))
    ok, X = solve(lib, body, A, B)
    assert ok
    # backward stable with partial pivoting (growth at most a few tens here):
    # the residual is m rounding errors of |A| |X|
    bound = 32.0 * m * EPS * (np.abs(A) @ np.abs(X) + np.abs(B))
    assert (np.abs(A @ X - B) <= bound).all()


def test_lu_zero_rows_move(lib, body):
    """A permutation: every pivot comes from a swap."""
    m = 9
    P = np.eye(m)[np.random.RandomState(2).permutation(m)]
    B = np.arange(2.0 * m).reshape(m, 2)
    ok, X = solve(lib, body, P, B)
    assert ok
    np.testing.assert_array_equal(X, P.T @ B)


def test_lu_singular(lib, body):
    for A in (np.zeros((1, 1)), np.ones((4, 4)), np.diag([1.0, 0.0, 2.0])):
        ok, _ = solve(lib, body, A, np.ones((len(A), 2)))
        assert not ok


def reference_solve(A, B):
    """Gaussian elimination with every product formed (no row is skipped)."""
    A, X = np.array(A, float), np.array(B, float)
    m = len(A)
    with np.errstate(invalid="ignore"):
        for c in range(m):
            for r in range(c + 1, m):
                f = A[r, c] * (1.0 / A[c, c])
                A[r, c + 1:] -= f * A[c, c + 1:]
                X[r] -= f * X[c]
        for r in range(m - 1, -1, -1):
            for k in range(r + 1, m):
                X[r] -= A[r, k] * X[k]
            X[r] /= A[r, r]
    return X


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("row", [0, 1, 3])
def test_lu_not_finite(lib, body, bad, row):
    """Observations out of each other's reach couple by zeros; a right-hand
    side that is not finite still reaches every row of its column, as the
    products by zero make it."""
    A = np.diag([2.0, 3.0, 4.0, 5.0])
    A[2, 3] = A[3, 2] = 1.0
    B = np.arange(8.0).reshape(4, 2)
    B[row, 1] = bad
    ok, X = solve(lib, body, A, B)
    assert ok
    want = reference_solve(A, B)
    np.testing.assert_array_equal(np.isfinite(X), np.isfinite(want))
    assert not np.isfinite(want[:, 1]).any()
    np.testing.assert_allclose(X[:, 0], want[:, 0], rtol=1e-15)


@pytest.mark.parametrize("m,p,q", [(1, 1, 1), (3, 2, 5), (64, 33, 17),
                                   (200, 32, 32)])
def test_gram(lib, body, m, p, q):
    rng = np.random.RandomState(m + p)
    X, Y = rng.uniform(-1, 1, (m, p)), rng.uniform(-1, 1, (m, q))
    got = np.empty((p, q))
    lib.gram(body, m, p, ptr(X), q, ptr(Y), ptr(got))
    assert (np.abs(got - X.T @ Y)
            <= 2.0 * m * EPS * (np.abs(X.T) @ np.abs(Y))).all()


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_bodies_agree(lib, seed):
    """Bit for bit, so that an analysis does not depend on the processor."""
    if not lib.has_body(1):
        pytest.skip("the processor has no AVX2")
    rng = np.random.RandomState(seed)
    m = 37
    A = rng.uniform(-1.0, 1.0, (m, m))
    A[rng.uniform(size=(m, m)) < 0.3] = 0.0  # zero multipliers too
    A += np.diag(rng.uniform(0.0, 2.0, m))
    B = rng.uniform(-1.0, 1.0, (m, 19))
    out = [solve(lib, body, A, B) for body in (0, 1)]
    assert out[0][0] and out[1][0]
    np.testing.assert_array_equal(out[0][1], out[1][1])
    C = [np.empty((m, 19)) for _ in range(2)]
    for body in (0, 1):
        lib.gram(body, m, m, ptr(A), 19, ptr(B), ptr(C[body]))
    np.testing.assert_array_equal(C[0], C[1])


@pytest.mark.parametrize("m", [1, 2, 3, 8, 33])
def test_is_diagonal(lib, m):
    R = np.diag(np.arange(m, dtype=float))  # a zero on the diagonal too
    assert lib.is_diagonal(m, ptr(R)) == 1
    R[0, 0] = np.nan
    assert lib.is_diagonal(m, ptr(R)) == 1
    for a, b in ((0, m - 1), (m - 1, 0), (m // 2, 0), (m - 1, m - 2)):
        for v in (1e-300, -1.0, np.nan, np.inf):
            if a == b or b < 0:
                continue
            Q = R.copy()
            Q[a, b] = v
            assert lib.is_diagonal(m, ptr(Q)) == 0, (a, b, v)
        if a != b and b >= 0:
            Q = R.copy()
            Q[a, b] = -0.0
            assert lib.is_diagonal(m, ptr(Q)) == 1
