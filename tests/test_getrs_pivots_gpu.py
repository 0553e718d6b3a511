"""Row interchanges of the single-system solve in any order: bzg_dgetrs follows ipiv as dlaswp does, also
where a row is interchanged with one above it (as no factorisation of this library does, but others may)."""
import numpy as np
import pytest

from gpu_util import ctx, dev, host, p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 5, 63, 64, 65, 130, 300, 1000])
@pytest.mark.parametrize("nrhs", [2, 70])
@pytest.mark.parametrize("kind", ["any", "above", "below", "same"])
def test_interchanges(n, nrhs, kind):
    rng = np.random.default_rng(n * 100 + nrhs)
    i = np.arange(n)
    q = {"any": rng.integers(0, n, n), "above": rng.integers(0, i + 1), "below": rng.integers(i, n),
         "same": np.full(n, n // 2)}[kind]
    B = rng.uniform(-1, 1, (n, nrhs))
    want = B.copy()
    for a, b in zip(i, q):
        want[[a, b]] = want[[b, a]]
    # the factors of the identity: the solution is the permuted right-hand side itself
    LU, piv, X = dev(np.eye(n)), dev((q + 1).astype(np.int32)), dev(B)
    ctx().call("bzg_dgetrs", n, nrhs, p(LU), n, p(piv), p(X), nrhs)
    assert np.array_equal(host(X), want)
