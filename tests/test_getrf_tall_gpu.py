"""Single-system LU of orders whose panels are taller than 4096, 8192 and 16384 rows (leaves of 4, 2 and 1
columns), with a partial last panel, guard columns and one zero column; checked on the GPU."""
import numpy as np
import pytest

from gpu_util import ctx, p, torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4161, 8257, 16449])
def test_tall(n):
    g = torch.Generator(device="cuda").manual_seed(n)
    lda, zero = n + 3, 70
    buf = torch.full((n, lda), 7.25, device="cuda", dtype=torch.float64)
    A = torch.rand((n, n), generator=g, device="cuda", dtype=torch.float64).mul_(2).sub_(1)
    A[:, zero] = 0.0
    buf[:, :n] = A
    piv = torch.zeros(n, device="cuda", dtype=torch.int32)
    info = torch.zeros(1, device="cuda", dtype=torch.int32)
    ctx().call("bzg_dgetrf", n, p(buf), lda, p(piv), p(info))
    assert int(info) == zero + 1 and bool((buf[:, n:] == 7.25).all())
    ip = piv.cpu().numpy() - 1
    assert np.all(ip >= np.arange(n)) and np.all(ip < n)
    perm = np.arange(n)
    for i, q in enumerate(ip):
        perm[i], perm[q] = perm[q], perm[i]
    v = torch.rand((n, 3), generator=g, device="cuda", dtype=torch.float64).mul_(2).sub_(1)
    PAv = (A @ v)[torch.from_numpy(perm).cuda()]
    absA = (A.abs_() @ v.abs())[torch.from_numpy(perm).cuda()]
    del A
    LU = buf[:, :n]
    L = torch.tril(LU, -1)
    assert float(L.abs().max()) <= 1.0
    U = torch.triu(LU)
    Uv = U @ v
    LUv = L @ Uv + Uv
    aUv = U.abs_() @ v.abs()
    bound = L.abs_() @ aUv + aUv
    # factorisation, and the products of the check themselves: gamma_n |L| |U| |v| each
    assert bool(((PAv - LUv).abs() <= (n + 2) * 2.0 ** -53 * (4 * bound + 2 * absA)).all())
