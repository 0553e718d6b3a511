"""The solves' division by a diagonal entry through its reciprocal: the quotient IEEE division gives, bit for
bit, over random operands, quotients near the ends of a binade, significands near 1 and 2, and the ends of the
exponent range (where the division itself is used)."""
import numpy as np
import pytest

from gpu_util import ctx, dev, host, p

pytestmark = pytest.mark.gpu


def operands(kind, size, rng):
    if kind == "random":
        return rng.uniform(1, 2, size) * 2.0 ** rng.integers(-40, 41, size)
    if kind == "near one":
        return 1.0 + rng.integers(-4096, 4096, size) * 2.0 ** -52
    if kind == "near two":
        return 2.0 - rng.integers(1, 4096, size) * 2.0 ** -52
    return rng.uniform(1, 2, size) * 2.0 ** rng.integers(-1074, 1024, size)  # "extreme"


@pytest.mark.parametrize("xs", ["random", "near one", "near two", "extreme"])
@pytest.mark.parametrize("ds", ["random", "near one", "near two", "extreme"])
@pytest.mark.parametrize("nrhs", [64, 65])
def test_quotients(xs, ds, nrhs):
    n = 1024
    rng = np.random.default_rng([len(xs), len(ds), nrhs])
    d = operands(ds, n, rng) * rng.choice([-1.0, 1.0], n)
    d[0] = 1.0  # (a factor is never zero here; the smallest may round to zero)
    d[d == 0.0] = 5e-324
    X = operands(xs, (n, nrhs), rng) * rng.choice([-1.0, 1.0], (n, nrhs))
    # quotients next to a power of two: the numerator from the divisor
    X[: n // 4] = (d[: n // 4, None] * (1.0 + rng.integers(-3, 4, (n // 4, nrhs)) * 2.0 ** -52))
    # a quotient that overflows would meet the zeros above the diagonal (inf * 0) in every other row
    with np.errstate(over="ignore", under="ignore"):
        X = np.where(np.isinf(X / d[:, None]), d[:, None], X)
    LU, piv, dX = dev(np.diag(d)), dev(np.arange(1, n + 1, dtype=np.int32)), dev(X)
    ctx().call("bzg_dgetrs", n, nrhs, p(LU), n, p(piv), p(dX), nrhs)
    with np.errstate(over="ignore", under="ignore"):
        want = X / d[:, None]
    got = host(dX)
    assert np.array_equal(got, want), np.argwhere(got != want)[:5]
