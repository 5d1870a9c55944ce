"""The block kinds of a network step (entry-wise, MFMA tile, long inner
dimension, split inner dimension with its sum) at the sizes where the choice
between them changes, and the step order when whole levels would not fit.
Against numpy's complex FP64 contraction; a product of inner length K is
held to (K + 8) rounding units of the same product of absolute values."""
import numpy as np
import pytest

from qaintensor import ops

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def crand(rng, *dims):
    return rng.standard_normal(dims) + 1j * rng.standard_normal(dims)


def split(n):
    """n as two legs (its largest divisor up to the square root first)."""
    d = max(x for x in range(1, int(n ** 0.5) + 1) if n % x == 0)
    return d, n // d


SIZES = [
    # elem: shortest, thin, up to 64 inner indices
    (1, 1, 1), (5, 3, 2), (3, 257, 7), (31, 33, 15), (17, 19, 64),
    # past elem: K = 65, and more than 2^22 products
    (17, 19, 65), (300, 800, 20),
    # long: from 512 inner indices, up to 16 entries, one to many blocks
    (1, 1, 511), (1, 1, 512), (4, 4, 1541), (16, 1, 1025), (1, 2, 70001),
    (1, 1, 1 << 21),
    # 17 and more entries over a long inner dimension: split tiles
    (17, 1, 512), (4, 5, 600), (70, 40, 1100),
    # 64 x 64 tiles
    (1024, 961, 66),
]


@pytest.mark.parametrize("m,n,k", SIZES)
@pytest.mark.parametrize("kfirst", [False, True])
def test_step_kinds(gpu_ctx, m, n, k, kfirst):
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    (m1, m2), (n1, n2), (k1, k2) = split(m), split(n), split(k)
    if kfirst:
        A, la = crand(rng, k1, m1, k2, m2), [1, -1, 2, -2]
        B, lb = crand(rng, k2, n1, n2, k1), [2, -3, -4, 1]
        am, bm = A.transpose(1, 3, 0, 2), B.transpose(3, 0, 1, 2)
    else:
        A, la = crand(rng, m1, k2, m2, k1), [-1, 2, -2, 1]
        B, lb = crand(rng, n1, k1, n2, k2), [-3, 1, -4, 2]
        am, bm = A.transpose(0, 2, 3, 1), B.transpose(1, 3, 0, 2)
    am = np.ascontiguousarray(am).reshape(m, k)
    bm = np.ascontiguousarray(bm).reshape(k, n)
    got = ops.contract_network([A, B], [la, lb], [1, 2])
    ref = (am @ bm).reshape(m1, m2, n1, n2)
    size = (np.abs(am) @ np.abs(bm)).reshape(ref.shape)
    assert got.shape == ref.shape
    assert np.all(np.abs(got - ref) <= (k + 8) * EPS * size)


def test_levels_that_would_not_fit_run_in_the_given_order(gpu_ctx):
    """Twelve independent outer-like products of 16 MiB each, every one
    closed to a number before the next in the given order: keeping the whole
    first level at once would take 192 MiB against about 16."""
    rng = np.random.default_rng(5)
    tensors, labels, order, ref = [], [], [], 1.0 + 0j
    for i in range(12):
        u, w = crand(rng, 1024, 2), crand(rng, 2, 1024)
        x, y = crand(rng, 1024), crand(rng, 1024)
        u, w, x, y = (t / np.linalg.norm(t) for t in (u, w, x, y))
        b = 3 * i
        tensors += [u, w, x, y]
        labels += [[b + 2, b + 1], [b + 1, b + 3], [b + 2], [b + 3]]
        order += [b + 1, b + 2, b + 3]
        ref *= x @ (u @ w) @ y
    got = complex(ops.contract_network(tensors, labels, order))
    # twelve factors, each two contractions of 1024 terms of unit vectors
    bound = sum(2 * (1024 + 8) * EPS for _ in range(12))
    scale = abs(ref)
    # |x (u w) y| is far below its unit bound, so bound each factor by it
    f = min(abs(tensors[4 * i + 2] @ (tensors[4 * i] @ tensors[4 * i + 1]) @
                tensors[4 * i + 3]) for i in range(12))
    assert abs(got - ref) <= bound / f * scale


def test_level_of_more_threads_than_a_grid_holds():
    """Three independent products of 37856 x 37856 entries (69 GB), all made
    before the first is closed: one level of more than 2^32 threads."""
    from qaintensor import Context
    rng = np.random.default_rng(6)
    d, tensors, labels, close, ref, f = 37856, [], [], [], 1.0 + 0j, 1.0
    for i in range(3):
        u, w = crand(rng, d, 2), crand(rng, 2, d)
        x, y = crand(rng, d), crand(rng, d)
        u, w, x, y = (t / np.linalg.norm(t) for t in (u, w, x, y))
        b = 10 * (i + 1)
        tensors += [u, w, x, y]
        labels += [[b + 1, i + 1], [i + 1, b + 2], [b + 1], [b + 2]]
        close += [b + 1, b + 2]
        ref *= (x @ u) @ (w @ y)
        f = min(f, abs((x @ u) @ (w @ y)))
    ctx = Context()
    got = complex(ops.contract_network(tensors, labels, [1, 2, 3] + close,
                                       ctx=ctx))
    ctx.close()
    # three factors, each two contractions of d terms of unit vectors
    assert abs(got - ref) <= 3 * 2 * (d + 8) * EPS / f * abs(ref)
