"""y = alpha*A^T*x + beta*y where its plan changes: x parts past the LDS tile,
rows walked one at a time and four at a time, row blocks that end early, split
K finished by the last workgroup (called twice, so tickets left uncleared would
show) and, through a captured graph, by the reduction kernel; exact integers,
NaN in the padding and between the vectors' elements."""
import numpy as np
import pytest
import torch

import eigen_amd as E
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,code", [(np.float32, E.F32), (np.float64, E.F64)])
@pytest.mark.parametrize("m,n,pad,incx,incy", [
    (1, 1, 0, 1, 1), (127, 3, 1, 2, 1), (129, 70, 0, 1, 3), (767, 33, 1, 1, 1), (1025, 257, 1, -1, 2), (4097, 300, 0, 1, 1),
    (8193, 17, 1, 3, -1), (16385, 64, 1, 1, 1), (40001, 9, 3, 1, 1), (300, 16390, 0, 1, 1)])
def test_gemv_t_exact(gpu, dtype, code, m, n, pad, incx, incy):
    A = O.fill((m + pad, n), dtype, 1, O.INT, -3, 3)
    A[m:] = np.nan
    x, y = O.fill((m, 1), dtype, 2, O.INT, -3, 3)[:, 0], O.fill((n, 1), dtype, 3, O.INT, -3, 3)[:, 0]
    want = 2.0 * (A[:m].astype(np.float64).T @ x) - y

    def spread(v, inc):
        s = np.full((len(v) - 1) * abs(inc) + 1, np.nan, dtype)
        s[::abs(inc)] = v if inc > 0 else v[::-1]
        return torch.from_numpy(s).cuda()

    a, dx, y0 = torch.from_numpy(A.reshape(-1, order="F").copy()).cuda(), spread(x, incx), spread(y, incy)
    dy = y0.clone()
    call = lambda s=None: E.gemv(code, 1, m, n, 2.0, a, m + pad, dx, incx, -1.0, dy, incy, stream=s)  # noqa: E731

    def check():
        torch.cuda.synchronize()
        got = dy.cpu().numpy()[::abs(incy)]
        assert np.array_equal((got if incy > 0 else got[::-1]).astype(np.float64), want)

    for _ in range(2):
        dy.copy_(y0)
        call()
        check()
    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.stream(s):
        call(s.cuda_stream)  # the stream's workspace exists before the capture
        torch.cuda.synchronize()
        g.capture_begin()
        call(s.cuda_stream)
        g.capture_end()
    for _ in range(2):
        dy.copy_(y0)
        torch.cuda.synchronize()
        g.replay()
        check()


@pytest.mark.parametrize("trans,m,n", [(1, 4099, 4097), (1, 300, 60000), (0, 8195, 4099)])
def test_gemv_past_the_cache_exact(gpu, trans, m, n):
    """Matrices that are read with the non-temporal hint (from 128 MB for A^T x, 256 MB for Ax)."""
    g = torch.Generator("cuda").manual_seed(1)
    a = torch.randint(-3, 4, (n, m), generator=g, device="cuda").double()
    x, y = (torch.randint(-3, 4, (k,), generator=g, device="cuda").double() for k in ((m, n) if trans else (n, m)))
    want = 2.0 * (a if trans else a.T) @ x - y
    E.gemv(E.F64, trans, m, n, 2.0, a.reshape(-1), m, x, 1, -1.0, y, 1)
    torch.cuda.synchronize()
    assert torch.equal(y, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("m,n,incx", [(2 ** 21 + 5, 1, 1), (2 ** 21 - 7, 3, 2), (40_000_003, 1, 1), (3_000_001, 4, 1),
                                      (4_200_000, 17, 1)])
def test_long_inner_products_exact(gpu, dtype, m, n, incx):
    """A^T x past 256 parts of x in LDS: several parts to a split, the sums of a
    block's rows kept between them; every sum is below 2^24."""
    g = torch.Generator("cuda").manual_seed(m)
    a = torch.zeros(n, m, dtype=dtype, device="cuda")
    x = torch.full(((m - 1) * incx + 1,), float("nan"), dtype=dtype, device="cuda")
    x[::incx] = torch.randint(-2, 3, (m,), generator=g, device="cuda").to(dtype)
    for j in range(n):
        a[j] = torch.randint(0, 2, (m,), generator=g, device="cuda").to(dtype)
    a[:, -1] = 1
    y0 = torch.arange(n, dtype=dtype, device="cuda")
    want = [2 * int((a[j].long() * x[::incx].long()).sum()) - j for j in range(n)]
    assert max(map(abs, want)) < 1 << 23
    code = E.F32 if dtype == torch.float32 else E.F64
    for _ in range(2):
        y = y0.clone()
        E.gemv(code, 1, m, n, 2.0, a.reshape(-1), m, x, incx, -1.0, y, 1)
        torch.cuda.synchronize()
        assert y.long().tolist() == want


@pytest.mark.parametrize("dtype,code", [(np.float32, E.F32), (np.float64, E.F64)])
@pytest.mark.parametrize("m", [1, 3, 64, 127, 128, 129, 255, 256, 257])
@pytest.mark.parametrize("n,pad,incx,incy", [(1, 0, 1, 1), (31, 1, 2, 1), (33, 3, -1, 2), (5000, 0, 1, -1), (16385, 1, 1, 1), (65537, 0, 2, 1)])
def test_gemv_t_short_rows_exact(gpu, dtype, code, m, n, pad, incx, incy):
    """Rows around one 1 KB load of a wave (128 FP64, 256 FP32 elements): each is
    followed by NaN, or by the next row, where it ends."""
    A = O.fill((m + pad, n), dtype, 1, O.INT, -3, 3)
    A[m:] = np.nan
    x, y = O.fill((m, 1), dtype, 2, O.INT, -3, 3)[:, 0], O.fill((n, 1), dtype, 3, O.INT, -3, 3)[:, 0]
    want = 2.0 * (A[:m].astype(np.float64).T @ x) - y
    dx = np.full((m - 1) * abs(incx) + 1, np.nan, dtype)
    dx[::abs(incx)] = x if incx > 0 else x[::-1]
    dy = np.full((n - 1) * abs(incy) + 1, np.nan, dtype)
    dy[::abs(incy)] = y if incy > 0 else y[::-1]
    a, dx, dy = (torch.from_numpy(v).cuda() for v in (A.reshape(-1, order="F").copy(), dx, dy))
    E.gemv(code, 1, m, n, 2.0, a, m + pad, dx, incx, -1.0, dy, incy)
    torch.cuda.synchronize()
    got = dy.cpu().numpy()[::abs(incy)]
    assert np.array_equal((got if incy > 0 else got[::-1]).astype(np.float64), want)


def test_gemv_t_past_one_grid(gpu):
    """More rows of A^T x than one launch of 32 to a workgroup holds (2^32 threads)."""
    n = 600_000_001
    a = torch.arange(n, device="cuda", dtype=torch.int32).remainder_(251).float()
    x = torch.full((1,), 3.0, device="cuda")
    y = torch.full((n,), float("nan"), device="cuda")
    E.gemv(E.F32, 1, 1, n, 2.0, a, 1, x, 1, 0.0, y, 1)
    torch.cuda.synchronize()
    assert torch.equal(a.mul_(6.0), y)
    y.fill_(float("nan"))
    E.gemm(E.F32, 0, 0, 1, n, 1, 0.5, x, 1, a, 1, 0.0, y, 1, prec=E.PREC_PLAIN)
    torch.cuda.synchronize()
    assert torch.equal(a.mul_(1.5), y)
