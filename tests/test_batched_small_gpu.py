"""Strided batches of products up to 32x32 and depth 64 on the one-wave kernel,
exactly (integer operands): one and two 16-wide blocks, every count of four-deep
steps, k shorter than a 16-byte run, a whole number of runs and every remainder,
padded leading dimensions and gaps between products (NaN there), beta = 0 over
NaN."""
import numpy as np
import pytest
import torch

import eigen_amd as E
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,code", [(np.float32, E.F32), (np.float64, E.F64)])
@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("m,n,k", [(1, 17, 1), (16, 16, 3), (17, 16, 5), (16, 17, 16), (32, 32, 17), (31, 30, 22), (32, 8, 25),
                                   (5, 32, 33), (29, 27, 47), (32, 32, 49), (20, 24, 62), (32, 31, 64)])
def test_one_wave_exact(gpu, dtype, code, ta, tb, m, n, k):
    count, pad = 37, 3
    ra, ca, rb, cb = (k, m, n, k) if ta and tb else (k, m, k, n) if ta else (m, k, n, k) if tb else (m, k, k, n)

    def batch(rows, cols, seed, gap):
        ld, x = rows + pad, np.full((count, cols * (rows + pad) + gap), np.nan, dtype)
        v = O.fill((count, cols * rows), dtype, seed, O.INT, -3, 3).reshape(count, cols, rows)
        x[:, :cols * ld].reshape(count, cols, ld)[:, :, :rows] = v
        return x, v.transpose(0, 2, 1).astype(np.float64), ld

    A, av, lda = batch(ra, ca, 1, 5)
    B, bv, ldb = batch(rb, cb, 2, 0)
    C, cv, ldc = batch(m, n, 3, 7)
    want = np.matmul(av.transpose(0, 2, 1) if ta else av, bv.transpose(0, 2, 1) if tb else bv)
    a, b = torch.from_numpy(A.ravel()).cuda(), torch.from_numpy(B.ravel()).cuda()
    for beta in (0.5, 0.0):
        start = C.copy()
        if beta == 0.0:
            start[:] = np.nan
        c = torch.from_numpy(start.ravel()).cuda()
        E.gemm_batched_strided(code, ta, tb, m, n, k, 2.0, a, lda, A.shape[1], b, ldb, B.shape[1], beta, c, ldc, C.shape[1],
                               count)
        torch.cuda.synchronize()
        got = c.cpu().numpy().reshape(C.shape)
        inner = got[:, :n * ldc].reshape(count, n, ldc)
        assert np.array_equal(inner[:, :, :m].transpose(0, 2, 1), 2.0 * want + (beta * cv if beta else 0.0))
        inner[:, :, :m] = 0
        start[:, :n * ldc].reshape(count, n, ldc)[:, :, :m] = 0
        assert np.array_equal(got, start, equal_nan=True)  # nothing else is written


@pytest.mark.parametrize("m", [17, 5])
def test_one_wave_past_one_grid(gpu, m):
    """More products than one launch of a wave each can hold (2^32 threads)."""
    count = (1 << 26) + 5
    a = torch.arange(count * m, device="cuda", dtype=torch.int32).remainder_(251).float()
    b = torch.arange(count, device="cuda", dtype=torch.int32).remainder_(13).float()
    c = torch.full((count * m,), float("nan"), device="cuda")
    E.gemm_batched_strided(E.F32, 0, 0, m, 1, 1, 2.0, a, m, m, b, 1, 1, 0.0, c, m, m, count)
    torch.cuda.synchronize()
    a.view(count, m).mul_(2.0 * b[:, None])
    assert torch.equal(a, c)
