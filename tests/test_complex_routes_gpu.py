"""Complex products that leave A in place do so only under the default planner,
outside a capture and where they have tiles enough: elsewhere they repack A and are, bit for bit, the real
product of the 2x2 block form that eh_gemm runs in the same way.  Operands are
not integers, and the in-place form's other order of summation shows in the
last bits (checked, so that the comparison means something)."""
import pytest
import torch

import eigen_amd as E

pytestmark = pytest.mark.gpu

M, N, K = 256, 200, 700


def operands(seed, M=M, N=N, K=K):
    g = torch.Generator("cuda").manual_seed(seed)
    a = torch.view_as_complex(torch.rand(K, M, 2, generator=g, dtype=torch.float64, device="cuda") - 0.5)  # column-major M x K
    b = torch.view_as_complex(torch.rand(N, K, 2, generator=g, dtype=torch.float64, device="cuda") - 0.5)
    a3 = torch.empty(2 * K, 2 * M, dtype=torch.float64, device="cuda")  # column-major 2M x 2K
    a3[0::2, 0::2], a3[0::2, 1::2] = a.real, a.imag
    a3[1::2, 0::2], a3[1::2, 1::2] = -a.imag, a.real
    return a.contiguous(), b.contiguous(), a3


def complex_product(a, b, c, stream=None):
    (K, M), N = a.shape, len(b)
    E.gemm_complex(E.F64, 0, 0, M, N, K, 1.0, a, M, b, K, 0.0, c, M, prec=E.PREC_PLAIN, stream=stream)


def real_product(a3, b, c, stream=None):
    (K, M), N = (x // 2 for x in a3.shape), len(b)
    E.gemm(E.F64, 0, 0, 2 * M, N, 2 * K, 1.0, a3, 2 * M, torch.view_as_real(b), 2 * K, 0.0, c, 2 * M,
           prec=E.PREC_PLAIN, stream=stream)


def both(a, b, a3):
    (K, M), N = a.shape, len(b)
    c, r = torch.zeros(N, M, dtype=torch.complex128, device="cuda"), torch.zeros(N, 2 * M, dtype=torch.float64, device="cuda")
    complex_product(a, b, c)
    real_product(a3, b, r)
    torch.cuda.synchronize()
    return torch.view_as_real(c).reshape(N, 2 * M), r


def test_other_planner(gpu):
    ops = operands(1)
    prev = E.lib().eh_get_tune_mode()
    try:
        E.set_tune_mode(E.TUNE_HEURISTIC)
        c, want = both(*ops)
        assert torch.equal(c, want)
        E.set_tune_mode(E.TUNE_MLP)
        c, _ = both(*ops)
        assert not torch.equal(c, want) and torch.allclose(c, want, rtol=0, atol=1e-12)
    finally:
        E.set_tune_mode(prev)


def test_captured(gpu):
    a, b, a3 = operands(2)
    c, r = torch.zeros(N, M, dtype=torch.complex128, device="cuda"), torch.zeros(N, 2 * M, dtype=torch.float64, device="cuda")
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        complex_product(a, b, c, s.cuda_stream)
        real_product(a3, b, r, s.cuda_stream)
        torch.cuda.synchronize()
        g.capture_begin()
        complex_product(a, b, c, s.cuda_stream)
        real_product(a3, b, r, s.cuda_stream)
        g.capture_end()
    for _ in range(3):
        c.zero_()
        r.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(torch.view_as_real(c).reshape(N, 2 * M), r)
        eager, _ = both(a, b, a3)
        assert torch.allclose(eager, r, rtol=0, atol=1e-12)


def test_few_tiles(gpu):
    """Two tiles of deep k: in place, one workgroup would add 64 parts each."""
    c, want = both(*operands(3, 64, 64, 2048))
    assert torch.equal(c, want)


def test_captured_after_one_eager_call(gpu):
    """The eager call, in place, grows the stream's workspace to what the captured
    one's split K needs (145 MB; its own slots take 48)."""
    m, n, k = 1603, 1483, 1537
    a, b, a3 = operands(4, m, n, k)
    assert E.config_info(E.plan(E.F64, 0, 0, 2 * m, n, 2 * k))[2] > 1
    c, s, g = torch.zeros(n, m, dtype=torch.complex128, device="cuda"), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    want = (b @ a).contiguous()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        complex_product(a, b, c, s.cuda_stream)
        torch.cuda.synchronize()
        assert torch.allclose(c, want, rtol=0, atol=1e-11)
        g.capture_begin()
        complex_product(a, b, c, s.cuda_stream)
        g.capture_end()
    for _ in range(2):
        c.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.allclose(c, want, rtol=0, atol=1e-11)
