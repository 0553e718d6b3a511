"""Single-system LU at the edges of its panels and leaves: orders around multiples of 64 (partial last
panels, whose rows must not reach past the matrix), around the leaf shapes' row counts, and the
right-hand-side counts where the triangular solve changes its method."""
import numpy as np
import pytest
import scipy.linalg as sl

from gpu_util import ctx, dev, host, p
from blaze_amd import solve as bsolve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [15, 16, 17, 63, 64, 65, 80, 127, 129, 255, 257, 300, 511, 513, 1023, 1025, 1535, 1540, 2047,
                               2050, 3071, 3075])
def test_factors_and_guard(n):
    """Pivots as LAPACK's, P A = L U to n u, and nothing written outside the matrix."""
    rng = np.random.default_rng(n)
    A = rng.uniform(-1, 1, (n, n))
    lda = n + 3
    buf = np.full((n + 64, lda), 7.25)  # 64 guard rows, 3 guard columns
    buf[:n, :n] = A
    d, piv, info = dev(buf), dev(np.zeros(n, np.int32)), dev(np.zeros(1, np.int32))
    ctx().call("bzg_dgetrf", n, p(d), lda, p(piv), p(info))
    out, ip = host(d), host(piv)
    assert host(info)[0] == 0
    assert np.all(out[n:] == 7.25) and np.all(out[:, n:] == 7.25)
    LU = out[:n, :n]
    _, pl = sl.lu_factor(A)
    assert np.array_equal(ip - 1, pl)
    perm = np.arange(n)
    for i, q in enumerate(ip - 1):
        perm[[i, q]] = perm[[q, i]]
    L, U = np.tril(LU, -1) + np.eye(n), np.triu(LU)
    # |P A - L U| <= gamma_n |L| |U| elementwise
    assert np.all(np.abs(A[perm] - L @ U) <= 2 * n * 2.0 ** -53 * (np.abs(L) @ np.abs(U)))


@pytest.mark.parametrize("n", [1, 63, 64, 65, 200, 577])
@pytest.mark.parametrize("nrhs", [1, 15, 16, 17, 64, 65])
def test_solve_widths(n, nrhs):
    rng = np.random.default_rng(n * 100 + nrhs)
    A, B = rng.uniform(-1, 1, (n, n)), rng.uniform(-1, 1, (n, nrhs))
    X, LU, ip, info = bsolve.gesv(ctx(), A, B)
    assert info == 0
    L, U = np.tril(LU, -1) + np.eye(n), np.triu(LU)
    perm = np.arange(n)
    for i, q in enumerate(ip - 1):
        perm[[i, q]] = perm[[q, i]]
    # backward error of the two substitutions and the factorisation: 3 gamma_n |L| |U| |x|
    bound = 3 * (n + 2) * 2.0 ** -53 * (np.abs(L) @ (np.abs(U) @ np.abs(X))) + 1e-300
    assert np.all(np.abs((B - A @ X)[perm]) <= bound + (n + 2) * 2.0 ** -53 * (np.abs(A) @ np.abs(X))[perm])


def test_zero_column_and_ties():
    """A zero column keeps its row and reports it; equal candidates take the lowest row; B untouched."""
    n = 130
    rng = np.random.default_rng(3)
    A = np.where(rng.uniform(size=(n, n)) < 0.5, -1.0, 1.0)  # every first candidate ties
    LU, ip, info = bsolve.getrf(ctx(), A)
    assert ip[0] == 1
    A = rng.uniform(-1, 1, (n, n))
    A[:, 70] = 0.0
    B = rng.uniform(-1, 1, (n, 5))
    X, _, ip, info = bsolve.gesv(ctx(), A, B)
    _, lp, linfo = sl.lapack.dgetrf(A)
    assert info == linfo == 71 and np.array_equal(ip - 1, lp) and np.array_equal(X, B)
