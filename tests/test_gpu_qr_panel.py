"""The Householder QR's panels of at most 512 rows (through the
preconditioned single SVD, which factors A and R^H): one and two rows per
thread, ragged last panels, the last panel taller than the tall-panel limit,
rank-deficient, zero and graded columns, and the zip-up split (QR of A^H).
Against LAPACK: every singular value within rows eps |A| and the factors'
product within 8 rows eps |A|."""
import numpy as np
import pytest

from qaintensor import ops

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def check(A):
    U, S, Vh = ops.svd(A)
    ref = np.linalg.svd(A, compute_uv=False)
    tol = max(A.shape) * EPS * np.linalg.norm(A)
    assert np.abs(S - ref).max() <= tol
    assert np.abs((U * S) @ Vh - A).max() <= 8 * tol


def crand(rng, *dims):
    return rng.standard_normal(dims) + 1j * rng.standard_normal(dims)


@pytest.mark.parametrize("m,n", [(512, 512), (541, 513), (515, 700),
                                 (530, 530)])
def test_preconditioned_svd(gpu_ctx, monkeypatch, m, n):
    monkeypatch.setenv("QTN_SVD_PRECOND", "1")
    rng = np.random.default_rng(m + n)
    check(crand(rng, m, n))
    A = crand(rng, m, n // 2) @ crand(rng, n // 2, n)
    A[:, 5::7] = 0
    check(A)
    check(crand(rng, m, n) * np.logspace(0, -9, n))
