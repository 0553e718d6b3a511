"""Triangular solves with infinities and NaN off the diagonal of the factors: within a block of 64 rows (32
where the solve recurses) a zero x(k) is skipped, as dtrsm does, so it meets neither."""
import numpy as np
import pytest

from blaze_amd import solve as bsolve
from gpu_util import ctx, dev, host, p

pytestmark = pytest.mark.gpu


def substitute(LU, B):
    """dtrsm's two substitutions (Left, NoTrans; unit lower, then upper), zeros skipped."""
    n, X = len(LU), B.copy()
    with np.errstate(all="ignore"):
        for c in range(X.shape[1]):
            for k in range(n):
                if X[k, c] != 0.0:
                    X[k + 1:, c] -= X[k, c] * LU[k + 1:, k]
            for k in reversed(range(n)):
                if X[k, c] != 0.0:
                    X[k, c] /= LU[k, k]
                    X[:k, c] -= X[k, c] * LU[:k, k]
    return X


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("n,nrhs", [(20, 1), (32, 16), (32, 65), (40, 3), (64, 1), (64, 17), (64, 65)])
@pytest.mark.parametrize("lower", [True, False])
def test_zero_entries_skip(value, n, nrhs, lower):
    """Small integers beside the special values: every other sum is exact."""
    rng = np.random.default_rng(n * 100 + nrhs)
    LU = np.where(rng.uniform(size=(n, n)) < 0.1, rng.integers(-2, 3, (n, n)), 0).astype(np.float64)
    np.fill_diagonal(LU, rng.choice([1.0, 2.0, -0.5], n))
    B = rng.integers(-4, 5, (n, nrhs)).astype(np.float64)
    # the special value stands in the column of an entry that stays zero in half of the right-hand sides
    k = 1 if lower else n - 2
    i = n - 1 if lower else 0
    LU[k, :k] = 0.0
    LU[k, k + 1:] = 0.0
    LU[i, k] = value
    B[k, ::2] = 0.0
    want = substitute(LU, B)
    assert np.all(np.isfinite(want[:, ::2])) and (nrhs == 1 or not np.all(np.isfinite(want[:, 1::2])))
    dLU, piv, X = dev(LU), dev(np.arange(1, n + 1, dtype=np.int32)), dev(B)
    ctx().call("bzg_dgetrs", n, nrhs, p(dLU), n, p(piv), p(X), nrhs)
    assert np.array_equal(host(X), want, equal_nan=True)


def test_infinite_entry():
    """A system with one infinite coefficient whose unknown is zero has a finite solution."""
    A = np.eye(20)
    A[0, 19] = np.inf
    B = np.eye(20)[:, :1]
    X, _, _, info = bsolve.gesv(ctx(), A, B)
    assert info == 0 and np.array_equal(X, B)
