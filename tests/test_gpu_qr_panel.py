"""The Householder QR's panels of at most 512 rows: one and two rows per
thread, ragged and short last panels, the last panel taller than the
tall-panel limit, rank-deficient, zero and graded columns.  Through the
preconditioned single SVD, which factors A and R^H (against LAPACK: every
singular value within rows eps |A|, the factors' product within 8 rows eps
|A|, the non-zero ones orthonormal to 1e-12), the zip-up's wide splits, which
factor A^H (against the oracle), and a layer of gates, which factors a batch
of uneven matrices (against the layer without the factorisation)."""
import numpy as np
import pytest

from oracle import qtn_oracle as O
from qaintensor import DeviceMPO, DeviceMPS, circuits as C, ops

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def check(A):
    U, S, Vh = ops.svd(A)
    ref = np.linalg.svd(A, compute_uv=False)
    tol = max(A.shape) * EPS * np.linalg.norm(A)
    assert np.abs(S - ref).max() <= tol
    assert np.abs((U * S) @ Vh - A).max() <= 8 * tol
    k = int(np.sum(S > 0))
    for Q in (U[:, :k], Vh[:k].conj().T):
        assert np.abs(Q.conj().T @ Q - np.eye(k)).max() <= 1e-12


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


# (bond dimensions of the middle of the chain): the splits have 2 k rows and
# three times the next bond's columns, so panels of 3 to 513 rows
@pytest.mark.parametrize("mid", [(3, 5, 9), (17, 21, 33), (61, 85, 86),
                                 (150, 170, 171)])
def test_zipup_splits_match_oracle(gpu_ctx, mid):
    n, cap, cutoff = 19, max(mid), 1e-8
    rng = np.random.default_rng(sum(mid))
    chis = [min(2 ** min(j, n - j), mid[j % 3]) for j in range(n + 1)]
    Bs = [crand(rng, chis[j], 2, chis[j + 1]) for j in range(n)]
    W = O.tfim_mpo(n, 1.0, rng.uniform(0.5, 1.5, n))
    Bc, _, _ = O.canonicalize(Bs)
    B_ref, lam_ref, nrm_ref = O.zipup(Bc, W, cutoff, cap)
    dev = DeviceMPS(n, cap, gpu_ctx)
    dev.set_sites([np.asfortranarray(b) for b in Bs])
    out = DeviceMPS(n, cap, gpu_ctx)
    nrm = dev.apply_mpo(DeviceMPO(W, gpu_ctx), cutoff, cap, out)
    assert abs(nrm - nrm_ref) <= 1e-10 * nrm_ref
    assert list(out.bond_dims()) == [1] + [b.shape[2] for b in B_ref]
    for j in range(1, n):
        assert np.abs(out.bond_spectrum(j) - lam_ref[j]).max() <= 1e-10
    for j in range(2, n + 1):
        B = out.site(j)
        v = B.reshape((B.shape[0], -1), order="F")
        assert np.abs(v @ v.conj().T - np.eye(B.shape[0])).max() <= 1e-12


@pytest.mark.parametrize("mid", [(33, 40, 37), (50, 65, 77), (130, 129, 150)])
def test_uneven_batches_match_without_qr(gpu_ctx, monkeypatch, mid):
    n, cap = 21, 2 * max(mid)
    rng = np.random.default_rng(sum(mid))
    chis = [min(2 ** min(j, n - j), mid[j % 3]) for j in range(n + 1)]
    ref = DeviceMPS(n, cap, gpu_ctx)
    ref.set_sites([np.asfortranarray(crand(rng, chis[j], 2, chis[j + 1]))
                   for j in range(n)])
    dev = DeviceMPS(n, cap, gpu_ctx)
    dev.copy_from(ref)
    sites = list(range(2, n, 2))
    gates = [C.haar_unitary(rng, 4) for _ in sites]
    k0, d0 = ref.apply_layer(sites, gates, 1e-8, max(mid))
    monkeypatch.setenv("QTN_JACOBI_PRECOND", "1")
    k1, d1 = dev.apply_layer(sites, gates, 1e-8, max(mid))
    assert np.array_equal(k0, k1)
    assert np.abs(d0 - d1).max() <= 1e-12
    for s in sites:
        assert np.abs(ref.bond_spectrum(s) -
                      dev.bond_spectrum(s)).max() <= 1e-12
        B = dev.site(s + 1)
        v = B.reshape((B.shape[0], -1), order="F")
        assert np.abs(v @ v.conj().T - np.eye(B.shape[0])).max() <= 1e-12
    f = abs(ref.overlap(dev)) ** 2 / (ref.norm2() * dev.norm2())
    assert abs(1.0 - f) <= 1e-10
