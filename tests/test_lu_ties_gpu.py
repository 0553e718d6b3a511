"""Pivot ties, at every step and among rows that earlier interchanges moved: the lowest row wins, as idamax
finds it.  The matrices (blocks of signs, their rows and columns scattered) are eliminated without
rounding, so the factors must equal a plain elimination's bit for bit."""
import numpy as np
import pytest

from blaze_amd import solve as bsolve
from gpu_util import ctx

pytestmark = pytest.mark.gpu


def sign_blocks(n, rng):
    """Row- and column-permuted block diagonal of regular 4 x 4 sign matrices."""
    A = np.zeros((n, n))
    for b in range(0, n, 4):
        S = np.zeros((4, 4))
        while abs(np.linalg.det(S)) < 0.5:
            S = rng.choice([-1.0, 1.0], (4, 4))
        A[b:b + 4, b:b + 4] = S
    return A[rng.permutation(n)][:, rng.permutation(n)]


def hadamard(n, rng):
    """Sylvester's matrix with random row and column signs: all candidates of every step tie."""
    H = np.ones((1, 1))
    while len(H) < n:
        H = np.block([[H, H], [H, -H]])
    return rng.choice([-1.0, 1.0], (n, 1)) * H * rng.choice([-1.0, 1.0], (1, n))


def eliminate(A):
    """dgetf2, column by column; only the rows that change."""
    A, n = A.copy(), len(A)
    piv = np.zeros(n, np.int32)
    for j in range(n):
        q = j + int(np.argmax(np.abs(A[j:, j])))  # the first of the largest
        piv[j] = q + 1
        A[[j, q]] = A[[q, j]]
        r = j + 1 + np.flatnonzero(A[j + 1:, j])
        A[r, j] /= A[j, j]
        A[r, j + 1:] -= np.outer(A[r, j], A[j, j + 1:])
    return A, piv


CASES = [(sign_blocks, n) for n in (4, 8, 64, 132, 200, 256, 300, 512)] + [(hadamard, n) for n in (16, 64, 128, 256, 512)]


@pytest.mark.parametrize("make,n", CASES + [(sign_blocks, 600), (sign_blocks, 1400), (sign_blocks, 2100),
                                            (sign_blocks, 3100), (hadamard, 1024)])
def test_getrf(make, n):
    A = make(n, np.random.default_rng(n))
    want, wp = eliminate(A)
    LU, piv, info = bsolve.getrf(ctx(), A)
    assert info == 0 and np.array_equal(piv, wp) and np.array_equal(LU, want)


def test_getrf_batched():
    As = [make(n, np.random.default_rng(n)) for make, n in CASES]
    LUs, pivs, infos = bsolve.getrf_batched(ctx(), As)
    assert np.all(infos == 0)
    for A, LU, piv in zip(As, LUs, pivs):
        want, wp = eliminate(A)
        assert np.array_equal(piv, wp) and np.array_equal(LU, want)
