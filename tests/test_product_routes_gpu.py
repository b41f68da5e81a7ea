"""Products that run the balanced kernel (asserted through eh_plan_kernel), all
op pairs and both types: exact with integer operands; and eh_gemm_noalloc bit for
bit as eh_gemm, eagerly and captured, with operands whose sums round."""
import ctypes as C

import numpy as np
import pytest
import torch

import eigen_amd as E
import oracle as O

pytestmark = pytest.mark.gpu
CODE = {np.float32: E.F32, np.float64: E.F64}
SHAPES = [(np.float64, 1000, 777, 1203), (np.float64, 130, 131, 9001), (np.float32, 779, 796, 1129),
          (np.float32, 130, 131, 20001)]


@pytest.fixture(autouse=True)
def default_planner(gpu):
    prev = E.lib().eh_get_tune_mode()
    E.set_tune_mode(E.TUNE_MLP)
    yield
    E.set_tune_mode(prev)


def dev(x):
    return torch.from_numpy(np.asarray(x).reshape(-1, order="F").copy()).cuda()


@pytest.mark.parametrize("ta", [0, 1])
@pytest.mark.parametrize("tb", [0, 1])
@pytest.mark.parametrize("dtype,m,n,k", SHAPES)
def test_balanced_exact(dtype, m, n, k, ta, tb):
    assert E.plan_kernel(CODE[dtype], ta, tb, m, n, k) == E.KERNEL_BALANCED
    A = O.fill((k, m) if ta else (m, k), dtype, 1, O.INT, -3, 3)
    B = O.fill((n, k) if tb else (k, n), dtype, 2, O.INT, -3, 3)
    C0 = O.fill((m, n), dtype, 3, O.INT, -3, 3)
    want = 2.0 * ((A.T if ta else A).astype(np.float64) @ (B.T if tb else B).astype(np.float64)) - C0
    a, b = dev(A), dev(B)
    for _ in range(2):  # twice: a ticket left uncleared would show
        c = dev(C0)
        E.gemm(CODE[dtype], ta, tb, m, n, k, 2.0, a, A.shape[0], b, B.shape[0], -1.0, c, m, prec=E.PREC_PLAIN)
        torch.cuda.synchronize()
        assert np.array_equal(c.cpu().numpy().reshape(n, m).T, want)


@pytest.mark.parametrize("dtype,m,n,k", SHAPES + [(np.float64, 96, 80, 112), (np.float32, 300, 1, 5000)])
def test_noalloc_same_bits(dtype, m, n, k):
    g = torch.Generator("cuda").manual_seed(1)
    t = torch.float32 if dtype == np.float32 else torch.float64
    a, b = (torch.rand(q, generator=g, dtype=t, device="cuda") - 0.5 for q in (m * k, k * n))
    one, zero = ((C.c_float if dtype == np.float32 else C.c_double)(v) for v in (1, 0))
    c, d = (torch.empty(m * n, dtype=t, device="cuda") for _ in range(2))

    def call(f, out, stream):
        E.check(f(CODE[dtype], 0, 0, m, n, k, C.byref(one), a.data_ptr(), m, b.data_ptr(), k, C.byref(zero),
                  out.data_ptr(), m, E.PREC_PLAIN, stream))

    L, s, graph = E.lib(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    call(L.eh_gemm, c, s.cuda_stream)
    call(L.eh_gemm_noalloc, d, s.cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(c, d)
    with torch.cuda.stream(s):
        graph.capture_begin()
        call(L.eh_gemm, c, s.cuda_stream)
        call(L.eh_gemm_noalloc, d, s.cuda_stream)
        graph.capture_end()
    for _ in range(2):
        c.zero_(), d.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, d) and bool(c.any())
