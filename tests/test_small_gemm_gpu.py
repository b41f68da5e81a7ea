"""The kernel for small plain products (32x32 tiles, eight waves sharing K),
exactly (integer operands) against the oracle's product: tile edges, k from one
element to past a step of every wave, padded and odd leading dimensions with NaN
in the padding, all op pairs; twice through a captured graph as well."""
import numpy as np
import pytest
import torch

import eigen_amd as E
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,code", [(np.float32, E.F32), (np.float64, E.F64)])
@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("m,n,k,pad", [(2, 2, 1, 0), (31, 33, 7, 1), (32, 32, 64, 0), (33, 65, 65, 3), (96, 80, 112, 0),
                                       (130, 7, 257, 2), (383, 384, 511, 1), (510, 512, 1023, 1)])
def test_small_exact(gpu, dtype, code, ta, tb, m, n, k, pad):
    ra, rb, ldc = (k if ta else m), (n if tb else k), m + pad
    A = O.fill((ra + pad, m if ta else k), dtype, 1, O.INT, -3, 3)
    B = O.fill((rb + pad, k if tb else n), dtype, 2, O.INT, -3, 3)
    A[ra:] = np.nan
    B[rb:] = np.nan
    C0 = O.fill((ldc, n), dtype, 3, O.INT, -3, 3)
    want = O.gemm_ref(bool(ta), bool(tb), 1.5, *map(np.asfortranarray, (A[:ra], B[:rb])), 0.5, np.asfortranarray(C0[:m]))
    flat = lambda x: torch.from_numpy(x.reshape(-1, order="F").copy()).cuda()  # noqa: E731
    a, b, c0 = flat(A), flat(B), flat(C0)
    c = c0.clone()
    call = lambda s=None: E.gemm(code, ta, tb, m, n, k, 1.5, a, ra + pad, b, rb + pad, 0.5, c, ldc,  # noqa: E731
                                 prec=E.PREC_PLAIN, stream=s)

    def check():
        torch.cuda.synchronize()
        got = c.cpu().numpy().reshape(n, ldc).T
        assert np.array_equal(got[:m].astype(np.float64), want)
        assert np.array_equal(got[m:], C0[m:])

    call()
    check()
    g, s = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.stream(s):
        torch.cuda.synchronize()
        g.capture_begin()
        call(s.cuda_stream)
        g.capture_end()
    for _ in range(2):
        c.copy_(c0)
        torch.cuda.synchronize()
        g.replay()
        check()
