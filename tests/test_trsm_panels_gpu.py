"""The real triangular solve's panel kernel at its edges: orders around the
64-row blocks and the 512-row panels, right-hand sides around the 16 columns
of a workgroup, every side / triangle / transpose arrangement, a leading
dimension past the kernel's 32-bit offsets, and NaN wherever nothing may be
read.

Bound: the forward error on well-conditioned triangles (diagonal 1..2,
off-diagonal entries O(1/order)) is at most 8 * order * u * ||X||_F against a
float64 solve; for FP64 the reference's own error adds the same again."""
import itertools

import numpy as np
import pytest
import torch

import eigen_amd as E
from helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu

U = {np.float32: 2.0 ** -24, np.float64: 2.0 ** -53}
ED = {np.float32: E.F32, np.float64: E.F64}
SIZES = [(63, 15), (64, 16), (65, 17), (128, 1), (129, 33), (200, 31), (511, 5), (512, 16), (513, 17), (577, 2),
         (1090, 18)]


def _triangle(rng, ka, dt, lower):
    a = rng.uniform(-1.0 / ka, 1.0 / ka, (ka, ka))
    a[np.arange(ka), np.arange(ka)] = rng.uniform(1.0, 2.0, ka) * np.where(np.arange(ka) % 2, 1.0, -1.0)
    i, j = np.indices((ka, ka))
    keep = i >= j if lower else i <= j
    t = np.where(keep, a, 0.0).astype(dt)
    return t, np.where(keep, t, np.nan).astype(dt)


def _check(dt, side, lower, trans, t, stored, lda, m, n, rng):
    ka = t.shape[0]
    A = np.full((lda, ka), np.nan, dtype=dt, order="F")
    A[:ka] = stored
    B = np.full((m + 3, n), np.nan, dtype=dt, order="F")
    B[:m] = rng.uniform(-1, 1, (m, n))
    dB = to_dev(B)
    E.trsm(ED[dt], E.LEFT if side == "L" else E.RIGHT, E.LOWER if lower else E.UPPER, E.OP_T if trans else E.OP_N,
           E.NON_UNIT, m, n, 1.5, to_dev(A), lda, dB, m + 3)
    got = from_dev(dB, B.shape)
    assert np.isnan(got[m:]).all(), "padding rows of B written"
    op = t.astype(np.float64).T if trans else t.astype(np.float64)
    rhs = 1.5 * B[:m].astype(np.float64)
    want = np.linalg.solve(op, rhs) if side == "L" else np.linalg.solve(op.T, rhs.T).T
    bound = (8 if dt == np.float32 else 16) * ka * U[dt] * np.linalg.norm(want)
    assert np.linalg.norm(got[:m] - want) <= bound, (side, lower, trans, m, n)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("ka,other", SIZES)
def test_panel_edges(gpu, dt, ka, other):
    rng = np.random.default_rng(ka)
    for side, lower, trans in itertools.product("LR", (True, False), (False, True)):
        t, stored = _triangle(rng, ka, dt, lower)
        m, n = (ka, other) if side == "L" else (other, ka)
        _check(dt, side, lower, trans, t, stored, ka + 1, m, n, rng)


@pytest.mark.parametrize("trans", [False, True])
def test_leading_dimension_past_32_bit_offsets(gpu, trans):
    ka, n, lda = 5, 3, (1 << 22) + 8
    rng = np.random.default_rng(5)
    t, stored = _triangle(rng, ka, np.float32, True)
    A = torch.full((ka * lda,), float("nan"), device="cuda")
    A.view(ka, lda)[:, :ka] = torch.from_numpy(stored.T.copy()).cuda()
    B = rng.uniform(-1, 1, (ka, n)).astype(np.float32)
    dB = to_dev(np.asfortranarray(B))
    E.trsm(E.F32, E.LEFT, E.LOWER, E.OP_T if trans else E.OP_N, E.NON_UNIT, ka, n, 1.0, A, lda, dB, ka)
    want = np.linalg.solve((t.T if trans else t).astype(np.float64), B.astype(np.float64))
    assert np.linalg.norm(from_dev(dB, B.shape) - want) <= 8 * ka * 2.0 ** -24 * np.linalg.norm(want)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("ka,other", [(2048, 3), (2049, 5), (2600, 18)])
def test_halves(gpu, dt, ka, other):
    """Systems of more than 2048 rows are halved first: every arrangement, a
    ragged last panel in either half, alpha applied once to both."""
    rng = np.random.default_rng(ka)
    for side, lower, trans in itertools.product("LR", (True, False), (False, True)):
        t, stored = _triangle(rng, ka, dt, lower)
        m, n = (ka, other) if side == "L" else (other, ka)
        _check(dt, side, lower, trans, t, stored, ka + 1, m, n, rng)
