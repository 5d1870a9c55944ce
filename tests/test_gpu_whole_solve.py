"""The inner solve of problems of one block pair (at most 64 columns) at the
widths where its path changes: one and two columns, odd widths, 32 and 33
(256 or 1024 threads), 63 and 64, tall and wide, rank-deficient, with zero
columns between others, and graded over ten decades.  Against LAPACK: every
singular value within rows eps |A|, factors orthonormal (non-zero ones) and
their product within 8 rows eps |A|."""
import numpy as np
import pytest

from qaintensor import ops

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def check(A):
    m, n = A.shape
    U, S, Vh = ops.svd(A)
    ref = np.linalg.svd(A, compute_uv=False)
    nrm = np.linalg.norm(A)
    tol = max(m, n, 64) * EPS * nrm
    assert np.abs(S - ref).max() <= tol
    assert np.abs((U * S) @ Vh - A).max() <= 8 * tol
    k = int(np.sum(S > 0))
    for Q in (U[:, :k], Vh[:k].conj().T):
        assert np.abs(Q.conj().T @ Q - np.eye(k)).max() <= 1e-12


@pytest.mark.parametrize("n", [1, 2, 3, 7, 16, 17, 31, 32, 33, 48, 63, 64])
@pytest.mark.parametrize("extra", [0, 5, 150])
def test_widths(gpu_ctx, n, extra):
    rng = np.random.default_rng(n * 10 + extra)
    A = rng.standard_normal((n + extra, n)) + \
        1j * rng.standard_normal((n + extra, n))
    check(A)
    check(np.ascontiguousarray(A.T))


@pytest.mark.parametrize("n", [5, 20, 32, 45, 64])
def test_deficient_zero_columns_and_graded(gpu_ctx, n):
    rng = np.random.default_rng(n)
    r = max(1, n // 3)
    L = rng.standard_normal((70, r)) + 1j * rng.standard_normal((70, r))
    R = rng.standard_normal((r, n)) + 1j * rng.standard_normal((r, n))
    check(L @ R)
    A = rng.standard_normal((70, n)) + 1j * rng.standard_normal((70, n))
    A[:, 1::3] = 0
    check(A)
    B = (rng.standard_normal((70, n)) + 1j * rng.standard_normal((70, n))) * \
        np.logspace(0, -10, n)
    check(B)
    check(np.eye(70, n, dtype=np.complex128))
