"""Graphs that hold a stream's workspace, and the workspace's growth around
them: integer operands, so every result is exact."""
import numpy as np
import pytest
import torch

import eigen_amd as E
import oracle as O

pytestmark = pytest.mark.gpu


def operands(m, n, k, seed):
    A, B = O.fill((m, k), np.float64, seed, O.INT, -3, 3), O.fill((k, n), np.float64, seed + 1, O.INT, -3, 3)
    dev = [torch.from_numpy(x.reshape(-1, order="F").copy()).cuda() for x in (A, B)]
    return dev, torch.from_numpy((A @ B).reshape(-1, order="F").copy()).cuda()


def product(m, n, k, ab, c, stream):
    E.gemm(E.F64, 0, 0, m, n, k, 1.0, ab[0], m, ab[1], k, 0.0, c, m, prec=E.PREC_PLAIN, stream=stream.cuda_stream)


def test_graph_outlives_growth(gpu):
    """A graph with a split-K product keeps its partial sums' buffer when later
    calls on its stream need a larger one, twice."""
    m, n, k = 130, 130, 20000
    assert E.config_info(E.plan(E.F64, 0, 0, m, n, k))[2] > 1
    ab, want = operands(m, n, k, 1)
    c = torch.zeros_like(want)
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        product(m, n, k, ab, c, s)
        torch.cuda.synchronize()
        g.capture_begin()
        product(m, n, k, ab, c, s)
        g.capture_end()
    for big in ((1000, 777, 1203), (1024, 1100, 9000)):
        bab, bwant = operands(*big, 5)
        bc = torch.zeros_like(bwant)
        with torch.cuda.stream(s):
            product(*big, bab, bc, s)
        torch.cuda.synchronize()
        assert torch.equal(bc, bwant)
        hold = torch.full((1 << 24,), float("nan"), dtype=torch.float64, device="cuda")  # takes freed memory
        for _ in range(2):
            c.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(c, want)
        assert torch.isnan(hold).all()


@pytest.mark.parametrize("before", [False, True])
def test_eager_call_beside_a_capture(gpu, before):
    """A product on one stream that needs that stream's first workspace, or a
    larger one, leaves the capture of another stream intact."""
    first = (1000, 777, 1203)
    ab, want = operands(96, 80, 112, 1)
    fab, fwant = operands(*first, 3)
    c, fc = torch.zeros_like(want), torch.zeros_like(fwant)
    s, t, g = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    if before:
        product(130, 130, 2000, *operands(130, 130, 2000, 7), t)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        g.capture_begin()
        product(96, 80, 112, ab, c, s)
        product(*first, fab, fc, t)
        g.capture_end()
    torch.cuda.synchronize()
    assert torch.equal(fc, fwant)
    for _ in range(2):
        c.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, want)


def test_replay_beside_eager_calls(gpu):
    """A graph replayed on another stream while the stream it was captured on
    runs products that need workspace: each keeps its own partial sums."""
    small, big = (130, 130, 20000), (1000, 777, 1203)
    ab, want = operands(*small, 1)
    bab, bwant = operands(*big, 3)
    c, bc = torch.zeros_like(want), torch.zeros_like(bwant)
    s, r, g = torch.cuda.Stream(), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        product(*small, ab, c, s)
        torch.cuda.synchronize()
        g.capture_begin()
        product(*small, ab, c, s)
        g.capture_end()
    for _ in range(30):
        c.zero_(), bc.zero_()
        torch.cuda.synchronize()
        for _ in range(4):
            with torch.cuda.stream(r):
                g.replay()
            product(*big, bab, bc, s)
        torch.cuda.synchronize()
        assert torch.equal(c, want) and torch.equal(bc, bwant)
