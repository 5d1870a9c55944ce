"""The rounds of problems wider than one block pair (65 columns and more) at
the sizes where they change path: two and three block pairs, odd ones, one
to eight 64-row chunks and more, wide and tall, rank-deficient, graded, with
zero columns, and batches through a layer of gates.  Against LAPACK: every
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
    tol = max(m, n, 64) * EPS * np.linalg.norm(A)
    assert np.abs(S - ref).max() <= tol
    assert np.abs((U * S) @ Vh - A).max() <= 8 * tol
    k = int(np.sum(S > 0))
    for Q in (U[:, :k], Vh[:k].conj().T):
        assert np.abs(Q.conj().T @ Q - np.eye(k)).max() <= 1e-12


def crand(rng, *dims):
    return rng.standard_normal(dims) + 1j * rng.standard_normal(dims)


@pytest.mark.parametrize("m,n", [
    (65, 65), (66, 65), (96, 96), (100, 630), (129, 128), (192, 130),
    (256, 256), (321, 77), (384, 200), (449, 320), (512, 129), (513, 100),
    (577, 66), (1100, 70), (70, 520)])
def test_sizes(gpu_ctx, m, n):
    check(crand(np.random.default_rng(m + n), m, n))


@pytest.mark.parametrize("m,n", [(90, 70), (140, 130), (300, 200)])
def test_deficient_zero_columns_and_graded(gpu_ctx, m, n):
    rng = np.random.default_rng(m * n)
    check(crand(rng, m, n // 3) @ crand(rng, n // 3, n))
    A = crand(rng, m, n)
    A[:, 3::5] = 0
    check(A)
    check(crand(rng, m, n) * np.logspace(0, -10, n))
    check(crand(rng, m, n) * np.logspace(-10, 0, n))
    check(np.eye(m, n, dtype=np.complex128))


@pytest.mark.parametrize("a,b", [(150, 150), (190, 140), (224, 130),
                                 (256, 256)])
@pytest.mark.parametrize("ng", [4, 5, 7])
def test_layers_of_tall_gates_match_single_gates(gpu_ctx, a, b, ng):
    """Two-site matrices of 300 to 512 rows, alternately wide and tall: a
    layer of them keeps its block pairs in registers from five square
    problems on, a gate alone takes three launches a round."""
    from qaintensor import DeviceMPS, circuits as C
    n = 2 * ng + 16
    dims = [min(2 ** min(j, n - j), a if j % 4 < 2 else b)
            for j in range(n + 1)]
    rng = np.random.default_rng(a + b + ng)
    ref = DeviceMPS(n, 256, gpu_ctx)
    ref.set_sites([np.asfortranarray(crand(rng, dims[j], 2, dims[j + 1]))
                   for j in range(n)])
    dev = DeviceMPS(n, 256, gpu_ctx)
    dev.copy_from(ref)
    sites = [9 + 2 * g for g in range(ng)]
    gates = [C.haar_unitary(rng, 4) for _ in sites]
    k, d = dev.apply_layer(sites, gates, 1e-8, 200)
    for g, s in enumerate(sites):
        k1, d1 = ref.apply_2q(s, gates[g], 1e-8, 200)[:2]
        assert k1 == k[g]
        assert abs(d1 - d[g]) <= 1e-12
        assert np.abs(ref.bond_spectrum(s) -
                      dev.bond_spectrum(s)).max() <= 1e-12
    f = abs(ref.overlap(dev)) ** 2 / (ref.norm2() * dev.norm2())
    assert abs(1.0 - f) <= 1e-10
    ref.free()
    dev.free()
