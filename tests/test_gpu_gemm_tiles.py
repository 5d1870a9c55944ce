"""The complex GEMMs at the sizes where the tile choice, the double-buffered
slices (16 inner indices) and the tile order change: one slice, a partial
last slice, fewer tiles than XCDs, tile counts that are no multiple of 8,
and sizes on both sides of the 64 x 64 rule.  An inner length K is held to
(K + 8) rounding units of the same product of absolute values."""
import ctypes

import numpy as np
import pytest

from qaintensor import _lib as L

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (33, 1, 16), (31, 65, 17), (64, 64, 15), (129, 65, 48),
         (320, 290, 33), (1000, 978, 31), (513, 1030, 18)]


@pytest.mark.parametrize("m,n,k", SIZES)
@pytest.mark.parametrize("ops", ["NN", "CN", "NC", "TT"])
@pytest.mark.parametrize("single", [False, True])
def test_gemm_tiles(gpu_ctx, m, n, k, ops, single):
    import torch
    dt = np.complex64 if single else np.complex128
    eps = np.finfo(dt).eps
    rng = np.random.default_rng(m + 2 * n + 3 * k)

    def mat(r, c):
        x = rng.standard_normal((r, c)) + 1j * rng.standard_normal((r, c))
        return np.asfortranarray(x.astype(dt))

    def op(x, o):
        return {"N": x, "T": x.T, "C": x.conj().T}[o]

    batch = 2 if m * n < 50000 else 1
    A = [mat(*((m, k) if ops[0] == "N" else (k, m))) for _ in range(batch)]
    B = [mat(*((k, n) if ops[1] == "N" else (n, k))) for _ in range(batch)]
    C = [mat(m, n) for _ in range(batch)]
    alpha, beta = 0.5 - 0.25j, -0.75 + 1j
    real = np.float32 if single else np.float64
    ptr = ctypes.POINTER(ctypes.c_float if single else ctypes.c_double)

    def up(xs):
        return torch.from_numpy(np.concatenate(
            [x.reshape(-1, order="F") for x in xs])).cuda()

    def dev(t):
        return ctypes.cast(t.data_ptr(), ptr)

    def host(z):
        a = np.array([z.real, z.imag], dtype=real)
        return a.ctypes.data_as(ptr), a

    dA, dB, dC = up(A), up(B), up(C)
    torch.cuda.synchronize()
    (pa, ka), (pb, kb) = host(alpha), host(beta)
    f = L.load().qtn_cgemm_dev if single else L.load().qtn_zgemm_dev
    L.check(f(gpu_ctx.handle, ops[0].encode(), ops[1].encode(), m, n, k, pa,
              dev(dA), A[0].shape[0], m * k, dev(dB), B[0].shape[0], k * n,
              pb, dev(dC), m, m * n, batch))
    gpu_ctx.sync()
    got = dC.cpu().numpy().reshape(batch, n, m).transpose(0, 2, 1)
    for g, a, b, c in zip(got, A, B, C):
        a, b = op(a, ops[0]).astype(np.complex128), \
            op(b, ops[1]).astype(np.complex128)
        ref = alpha * (a @ b) + beta * c
        size = np.abs(alpha) * (np.abs(a) @ np.abs(b)) + \
            np.abs(beta) * np.abs(c)
        # complex products double the terms of every inner index
        assert np.all(np.abs(g - ref) <= (2 * k + 8) * eps * size)


@pytest.mark.parametrize("m", [2**29 - 33, 2**29 + 33])
def test_more_rows_than_small_tiles_can_launch(m):
    """An outer product of a long column, on both sides of the 2^24 small
    tiles that a grid's first dimension holds."""
    import torch
    from qaintensor import Context
    n = 2
    A = torch.randn(m, dtype=torch.complex64, device="cuda")
    B = torch.tensor([0.5 - 2j, -1 + 0.25j], dtype=torch.complex64).cuda()
    C = torch.zeros(n, m, dtype=torch.complex64, device="cuda")
    one = np.array([1.0, 0.0], dtype=np.float32)
    zero = np.zeros(2, dtype=np.float32)
    ptr = ctypes.POINTER(ctypes.c_float)

    def dev(t):
        return ctypes.cast(t.data_ptr(), ptr)

    torch.cuda.synchronize()
    ctx = Context()
    L.check(L.load().qtn_cgemm_dev(
        ctx.handle, b"N", b"N", m, n, 1, one.ctypes.data_as(ptr), dev(A), m,
        0, dev(B), 1, 0, zero.ctypes.data_as(ptr), dev(C), m, 0, 1))
    ctx.sync()
    # one complex product per entry
    for j in range(n):
        err = torch.abs(C[j] - A * B[j])
        assert bool(torch.all(err <= 10 * 2.0**-23 * torch.abs(A) *
                              abs(complex(B[j]))))
        del err
    ctx.close()
    del A, B, C
    torch.cuda.empty_cache()
