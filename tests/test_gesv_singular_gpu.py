"""bzg_dgesv on a singular matrix reports info and needs nothing else: no right-hand sides and no scratch
for the solve.  The same calls on a regular matrix are errors, and the context works after them."""
import numpy as np
import pytest

import blaze_amd as bz
from gpu_util import ctx, dev, host, p

pytestmark = pytest.mark.gpu

HUGE = 1 << 36  # right-hand sides whose scratch (512 GB a row) cannot be had


def call(n, singular, nrhs, B):
    rng = np.random.default_rng(n)
    A = rng.uniform(-1, 1, (n, n)) + n * np.eye(n)
    if singular:
        A[:, n // 2] = 0.0
    piv, info = dev(np.zeros(n, np.int32)), dev(np.full(1, -7, np.int32))
    dA = dev(A)
    ctx().call("bzg_dgesv", n, nrhs, p(dA), n, p(piv), B, nrhs, p(info))
    return int(host(info)[0])


@pytest.mark.parametrize("n", [1, 30, 100])
@pytest.mark.parametrize("what", ["no B", "no memory"])
def test_singular(n, what):
    B = dev(np.full(8, 2.5))
    nrhs, ptr = (3, None) if what == "no B" else (HUGE, p(B))
    assert call(n, True, nrhs, ptr) == n // 2 + 1
    with pytest.raises(bz.BlazeGpuError):
        call(n, False, nrhs, ptr)
    X = dev(np.eye(n))
    assert call(n, False, n, p(X)) == 0  # the context still solves
    assert np.all(np.isfinite(host(X))) and np.array_equal(host(B), np.full(8, 2.5))
