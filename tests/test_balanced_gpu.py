"""The balanced product kernel: products whose tiles are cut between
workgroups, complex A read in place, and triangular products, exactly (integer
operands, every sum below 2^24 in FP32) against the oracle.  The shapes put
tile edges, k remainders and cuts at different places: fewer units than
workgroups, several cuts in a tile, several tiles in a run, one k slice.  Each
shape runs twice on one stream, so tickets left uncleared would show, and once
more from a captured graph, which takes the form without tickets."""
import numpy as np
import pytest
import torch

import eigen_amd as E
import oracle as O

pytestmark = pytest.mark.gpu
TYPES = {np.float32: E.F32, np.float64: E.F64}


def dev(x):
    return torch.from_numpy(np.asarray(x).reshape(-1, order="F").copy()).cuda()


def host(t, rows, cols):
    return t.cpu().numpy().reshape(cols, rows).T


def every_way(call, out, start):
    """call() eagerly twice, then (after one call on its stream, as the
    library asks of callers that capture) through a graph; out after each."""
    got = []
    for _ in range(2):
        out.copy_(start)
        call(0)
        torch.cuda.synchronize()
        got.append(out.clone())
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        call(s.cuda_stream)
        torch.cuda.synchronize()
        g.capture_begin()
        call(s.cuda_stream)
        g.capture_end()
    for _ in range(2):
        out.copy_(start)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got.append(out.clone())
    return got


# shapes the planner's rule sends to the balanced kernel: FP64 64x64 tiles, two
# and three workgroups per CU, FP32 64x64 and (large) 128x128 tiles
@pytest.mark.parametrize("dtype,ta,tb,m,n,k", [
    (np.float64, True, False, 1000, 777, 1203), (np.float64, False, False, 2049, 701, 2999),
    (np.float64, False, True, 1573, 721, 1985), (np.float32, False, True, 779, 796, 1129),
    (np.float32, True, False, 1645, 1384, 2731), (np.float64, True, True, 3140, 3448, 515)])
def test_plain(gpu, dtype, ta, tb, m, n, k):
    A = O.fill((k, m) if ta else (m, k), dtype, 1, O.INT, -3, 3)
    B = O.fill((n, k) if tb else (k, n), dtype, 2, O.INT, -3, 3)
    C0 = O.fill((m, n), dtype, 3, O.INT, -3, 3)
    a, b, c0 = dev(A), dev(B), dev(C0)
    c = torch.empty_like(c0)
    for got in every_way(lambda s: E.gemm(TYPES[dtype], int(ta), int(tb), m, n, k, 2.0, a, A.shape[0], b, B.shape[0], -1.0,
                                          c, m, prec=E.PREC_PLAIN, stream=s), c, c0):
        want = 2.0 * (A.T if ta else A).astype(np.float64) @ (B.T if tb else B).astype(np.float64) - C0
        assert np.array_equal(host(got, m, n), want)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("opa", [0, 1, 2])
@pytest.mark.parametrize("m,n,k,pad", [(1, 2, 1, 0), (31, 33, 7, 1), (33, 65, 17, 2), (200, 130, 301, 3),
                                       (1025, 1100, 65, 1)])
def test_complex_a_in_place(gpu, dtype, opa, m, n, k, pad):
    lda = (m if opa == 0 else k) + pad
    def ints(shape, seed):
        return O.fill(shape, dtype, seed, O.INT, -3, 3) + 1j * O.fill(shape, dtype, seed + 1, O.INT, -3, 3)
    A, B, C0 = ints((lda, k if opa == 0 else m), 1), ints((k, n), 3), ints((m, n), 5)
    A[m if opa == 0 else k:] = np.nan  # padding rows are not read
    op = A[:m] if opa == 0 else (A[:k].T if opa == 1 else A[:k].conj().T)
    want = (2 - 1j) * (op.astype(np.complex128) @ B.astype(np.complex128)) + 3.0 * C0
    ct = np.complex64 if dtype == np.float32 else np.complex128
    a, b, c0 = dev(A.astype(ct)), dev(B.astype(ct)), dev(C0.astype(ct))
    c = torch.empty_like(c0)
    for got in every_way(lambda s: E.gemm_complex(TYPES[dtype], opa, 0, m, n, k, 2 - 1j, a, lda, b, k, 3.0, c, m,
                                                  prec=E.PREC_PLAIN, stream=s), c, c0):
        assert np.array_equal(host(got, m, n), want)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("side,uplo,op", [(s, u, o) for s in "LR" for u in "LU" for o in "NT"])
@pytest.mark.parametrize("order,other,unit", [(1, 3, 0), (63, 1, 1), (65, 130, 0), (130, 64, 1), (700, 333, 0),
                                              (2050, 70, 1)])
def test_triangular(gpu, dtype, side, uplo, op, order, other, unit):
    ld = order + 1
    T = O.fill((ld, order), dtype, 1, O.INT, -3, 3)
    keep = np.tri(order, dtype=bool) if uplo == "L" else np.tri(order, dtype=bool).T
    if unit:
        keep = keep & ~np.eye(order, dtype=bool)
    D = np.where(keep, T[:order], 0) + (np.eye(order) if unit else 0)
    T[:order][~keep] = np.nan  # the other triangle and a unit diagonal are not read
    T[order] = np.nan
    m, n = (order, other) if side == "L" else (other, order)
    B = O.fill((m, n), dtype, 2, O.INT, -3, 3)
    D = (D if op == "N" else D.T).astype(np.float64)
    want = -2.0 * (D @ B if side == "L" else B @ D)
    a, b0 = dev(T), dev(B)
    b = torch.empty_like(b0)
    for got in every_way(lambda s: E.trmm(TYPES[dtype], E.LEFT if side == "L" else E.RIGHT,
                                          E.LOWER if uplo == "L" else E.UPPER, "NT".index(op),
                                          E.UNIT if unit else E.NON_UNIT, m, n, -2.0, a, ld, b, m, stream=s), b, b0):
        assert np.array_equal(host(got, m, n), want)
