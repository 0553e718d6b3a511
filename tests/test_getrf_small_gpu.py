"""Single-system LU and solves at the smallest orders, and at the last rows of a partial panel, where a narrower
leaf factors and a solve changes its method: factors exact against an elimination in the same order, guard rows
and columns untouched."""
import numpy as np
import pytest

from gpu_util import ctx, dev, host, p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 6, 7, 8, 9, 24, 25, 65, 71, 72, 73, 129, 136])
@pytest.mark.parametrize("nrhs", [1, 17])
def test_small(n, nrhs):
    rng = np.random.default_rng(n)
    L = np.tril(rng.integers(-1, 2, (n, n)), -1) / 2 + np.eye(n)  # |l| < 1: no ties with the diagonal
    U = np.triu(rng.integers(-3, 4, (n, n)), 1) + np.diag(rng.choice([1.0, -2.0, 4.0], n))
    order = rng.permutation(n)
    A = (L @ U)[order]  # exact: every pivot and product is a short dyadic number
    X = rng.integers(-4, 5, (n, nrhs)).astype(np.float64)
    buf = np.full((n + 2, n + 3), 7.25)
    buf[:n, :n] = A
    d, piv, info, dX = dev(buf), dev(np.zeros(n, np.int32)), dev(np.zeros(1, np.int32)), dev(A @ X)
    ctx().call("bzg_dgesv", n, nrhs, p(d), n + 3, p(piv), p(dX), nrhs, p(info))
    out, ip = host(d), host(piv) - 1
    perm = np.arange(n)
    for i, q in enumerate(ip):
        assert i <= q < n
        perm[[i, q]] = perm[[q, i]]
    assert host(info)[0] == 0 and np.all(out[n:] == 7.25) and np.all(out[:, n:] == 7.25)
    assert np.array_equal(order[perm], np.arange(n))
    assert np.array_equal(out[:n, :n], np.tril(L, -1) + U)
    if n <= 9:  # the substitutions' intermediate values stay exact
        assert np.array_equal(host(dX), X)
    else:
        assert np.all(np.abs(A @ host(dX) - A @ X) <= 3 * (n + 2) * 2.0 ** -53
                      * ((np.abs(L) @ (np.abs(U) @ np.abs(host(dX))))[np.argsort(perm)] + np.abs(A @ X)))
