"""BF16x3 products whose partial sums only grow: the error stays that of the
24-bit operands at every inner length, against numpy in FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 2k embedded inner indices in steps of 32, two steps to an FP64 addition:
# one step, an odd and an even number of them, a remainder, a long sum; rows
# and columns at the edges of the 128 x 128 tiles and over several of them
@pytest.mark.parametrize("m,n,k", [
    (1, 1, 1), (63, 127, 16), (64, 128, 48), (65, 129, 33), (200, 5, 500),
    (130, 260, 4096),
])
@pytest.mark.parametrize("op", ["N", "C"])
def test_long_sums_keep_the_operands_precision(gpu_ctx, op, m, n, k):
    from qaintensor import ops
    rng = np.random.default_rng(m + 10 * n + 100 * k)

    def pos(*shape):
        return (rng.uniform(0.5, 1.0, shape)
                + 1j * rng.uniform(0.5, 1.0, shape))

    A = pos(m, k) if op == "N" else pos(k, m)
    B = pos(k, n)
    opA = A if op == "N" else A.conj().T
    C = ops.zgemm_bf16x3(A, B, op, ctx=gpu_ctx)
    # operands and dropped terms: 4 * 2^-24 of sum |a| |b|; 12 FP32 additions
    # between two FP64 ones, each within 2 * 2^-24 of the partial sum
    mag = 2 * (np.abs(opA) @ np.abs(B))
    assert np.all(np.abs(C - opA @ B) <= 28 * 2.0**-24 * mag)
