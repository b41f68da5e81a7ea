"""The dense-product work that the library's performance is measured on.

Each case is one call (or one replay of a batch) through the package's public
entry points on operands resident in HBM, as a program that links the library
in Eigen's or BLAS's place makes it.  `listed()` gives fixed cases, `draw()`
more of the same ranges; see the comments at each for what they stand for.

    prepare(case, seed)  operands (from the seed alone), handles, outputs
    run(state)           one pass; returns the whole outputs
    work(case)           bytes and flops one pass cannot do without
    exact(case, seed)    the outputs in 64-bit arithmetic by torch alone

Matrices are column-major and dense (leading dimension = rows) in flat
buffers; a matrix with r rows and c columns is `buffer.view(c, r).T`.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import eigen_amd as E

DEV = "cuda:0"
REAL = {"f32": torch.float32, "f64": torch.float64}
CPLX = {"f32": torch.complex64, "f64": torch.complex128}
HALF = {"bf16": torch.bfloat16, "f16": torch.float16}
CODE = {"f32": E.F32, "f64": E.F64}
OPS = {"N": E.OP_N, "T": E.OP_T, "C": E.OP_C}
PRECS = {"plain": E.PREC_PLAIN, "split2": E.PREC_SPLIT2, "split3": E.PREC_SPLIT3}


def listed():
    return [
        # The smallest calls: an Eigen program's everyday small dynamic matrices,
        # one product per call.  Latency, launches and host work are all there is.
        dict(name="gemm_f32_small", kind="gemm", dtype="f32", opa="N", opb="N", m=96, n=80, k=112,
             alpha=1.5, beta=0.5, prec="plain"),
        # Ordinary products with ragged sizes, both real types, transposed operands:
        # normal equations, projections, covariance-like products.
        dict(name="gemm_f64_ordinary", kind="gemm", dtype="f64", opa="T", opb="N", m=1000, n=777, k=1203,
             alpha=1.0, beta=0.0, prec="plain"),
        dict(name="gemm_f32_ordinary", kind="gemm", dtype="f32", opa="N", opb="T", m=2500, n=1801, k=2100,
             alpha=1.0, beta=1.0, prec="plain"),
        # The dgemm drop-in at a size that fills the chip (the benchmark's dgemm leg).
        dict(name="gemm_f64_large", kind="gemm", dtype="f64", opa="N", opb="N", m=4096, n=4096, k=4096,
             alpha=1.5, beta=0.5, prec="plain"),
        # The benchmark's headline: FP32 sgemm on the BF16 matrix cores, three
        # terms per operand, entries over sixteen binades.
        dict(name="gemm_split3_large", kind="gemm", dtype="f32", opa="N", opb="N", m=8192, n=8192, k=8192,
             alpha=1.0, beta=0.0, prec="split3"),
        # 16-bit inputs, FP32 result (the sbgemm redirect and half matrices).
        dict(name="gemm_bf16_large", kind="half", dtype="bf16", opa="N", opb="N", m=8192, n=8192, k=8192,
             alpha=1.0, beta=0.0),
        # Triangular solve with many right-hand sides, in place, at an ordinary
        # odd order: what follows every Cholesky or LU factorisation.
        dict(name="trsm_f64", kind="trsm", dtype="f64", side="L", uplo="L", op="N", m=1000, n=600),
        # The other level-3 routines: triangular product from the right.
        dict(name="trmm_f32", kind="level3", routine="trmm", dtype="f32", side="R", uplo="U", op="T", m=1500, n=1100),
        # Complex product with a conjugated operand.
        dict(name="gemm_c128_ordinary", kind="complex", dtype="f64", opa="C", opb="N", m=1024, n=700, k=1500),
        # Matrix-vector product: one pass over a matrix in HBM.
        dict(name="gemv_f64", kind="gemv", dtype="f64", field="real", op="T", m=6000, n=4001),
        # Arrays of one fixed small size (the benchmark's strided leg).
        dict(name="strided_f64_16", kind="strided", dtype="f64", opa="N", opb="N", m=16, n=16, k=16, count=20000),
        # Thousands of small uneven products in one replayed graph (the
        # benchmark's batched leg): half FP32, half FP64.
        dict(name="grouped_uneven", kind="grouped", count=20000, lo=4, hi=256, shapes=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["small", "ordinary", "large", "split", "half", "trsm", "level3", "complex", "gemv", "strided",
                       "grouped"])
    dtype = rng.choice(["f32", "f64"])
    if kind in ("small", "ordinary", "large"):
        lo, hi = {"small": (16, 384), "ordinary": (384, 3000), "large": (3000, 5000)}[kind]
        return dict(kind="gemm", dtype=dtype, opa=rng.choice("NT"), opb=rng.choice("NT"), m=_log(rng, lo, hi),
                    n=_log(rng, lo, hi), k=_log(rng, lo, hi), alpha=rng.choice([1.0, 1.5]),
                    beta=rng.choice([0.0, 0.5, 1.0]), prec="plain")
    if kind == "split":
        return dict(kind="gemm", dtype="f32", opa=rng.choice("NT"), opb=rng.choice("NT"), m=_log(rng, 1024, 8192),
                    n=_log(rng, 1024, 8192), k=_log(rng, 1024, 8192), alpha=1.0, beta=rng.choice([0.0, 1.0]),
                    prec=rng.choice(["split2", "split3"]))
    if kind == "half":
        # leading dimensions multiples of 8 as often as not
        step = rng.choice([1, 8])
        dim = lambda: max(step, _log(rng, 512, 8192) // step * step)  # noqa: E731
        return dict(kind="half", dtype=rng.choice(["bf16", "f16"]), opa=rng.choice("NT"), opb=rng.choice("NT"),
                    m=dim(), n=dim(), k=dim(), alpha=1.0, beta=rng.choice([0.0, 1.0]))
    if kind == "trsm":
        return dict(kind="trsm", dtype=dtype, side=rng.choice("LR"), uplo=rng.choice("UL"), op=rng.choice("NT"),
                    m=_log(rng, 64, 3000), n=_log(rng, 64, 3000))
    if kind == "level3":
        return dict(kind="level3", routine=rng.choice(["trmm", "symm", "syrk"]), dtype=dtype, side=rng.choice("LR"),
                    uplo=rng.choice("UL"), op=rng.choice("NT"), m=_log(rng, 64, 3000), n=_log(rng, 64, 3000))
    if kind == "complex":
        return dict(kind="complex", dtype=dtype, opa=rng.choice("NTC"), opb=rng.choice("NTC"), m=_log(rng, 128, 2048),
                    n=_log(rng, 128, 2048), k=_log(rng, 128, 2048))
    if kind == "gemv":
        return dict(kind="gemv", dtype=dtype, field=rng.choice(["real", "real", "complex"]), op=rng.choice("NT"),
                    m=_log(rng, 256, 16384), n=_log(rng, 256, 16384))
    if kind == "strided":
        m, n, k = (_log(rng, 2, 64) for _ in range(3))
        room = 2e8 / (8 * (m * k + k * n + m * n))
        return dict(kind="strided", dtype=dtype, opa=rng.choice("NT"), opb=rng.choice("NT"), m=m, n=n, k=k,
                    count=_log(rng, 500, max(1000, min(100000, room))))
    return dict(kind="grouped", count=_log(rng, 1000, 20000), lo=4, hi=rng.choice([64, 128, 256]),
                shapes=rng.randrange(1 << 20))


# ---- operands ---------------------------------------------------------------------

def _uniform(g, n, dtype):
    if dtype.is_complex:
        real = torch.float64 if dtype == torch.complex128 else torch.float32
        return torch.view_as_complex(torch.rand(n, 2, generator=g, dtype=real, device=DEV) * 2 - 1)
    if dtype in (torch.float32, torch.float64):
        return torch.rand(n, generator=g, dtype=dtype, device=DEV) * 2 - 1
    return (torch.rand(n, generator=g, device=DEV) * 2 - 1).to(dtype)


def _wide(g, n):
    """FP32 entries sign * U(1, 2) * 2^U(-8, 8): the split products' inputs."""
    u = torch.rand(n, 2, generator=g, device=DEV)
    s = torch.randint(0, 2, (n,), generator=g, device=DEV) * 2 - 1
    return (1 + u[:, 0]) * torch.exp2(u[:, 1] * 16 - 8) * s


def _triangle(g, order, dtype):
    """A square matrix whose triangles are well conditioned: diagonal 2, the
    other entries U[-1/order, 1/order]."""
    a = _uniform(g, order * order, dtype) / order
    a.view(order, order).diagonal().fill_(2)
    return a


def _stored(op, rows, cols):
    """Stored rows and columns of a matrix whose op() is rows x cols."""
    return (rows, cols) if op == "N" else (cols, rows)


def _batch_shapes(case):
    rng = np.random.default_rng(case["shapes"])
    lo, hi = math.log(case["lo"]), math.log(case["hi"])
    return np.rint(np.exp(rng.uniform(lo, hi, size=(case["count"], 3)))).astype(np.int64)


def _inputs(case, seed):
    """Operands A, B and the result's initial value C, flat column-major."""
    g = torch.Generator(DEV)
    g.manual_seed(seed)
    kind = case["kind"]
    if kind == "grouped":  # per type: the operands of its products one after another
        out = {}
        half = case["count"] // 2
        for name, dims in (("f32", _batch_shapes(case)[:half]), ("f64", _batch_shapes(case)[half:])):
            m, n, k = dims.T
            out[name] = tuple(_uniform(g, int(x.sum()), REAL[name]) for x in (m * k, k * n)) + (
                torch.zeros(int((m * n).sum()), dtype=REAL[name], device=DEV),)
        return out
    m, n, dtype = case["m"], case["n"], case["dtype"]
    if kind in ("gemm", "half", "complex", "strided"):
        k, count = case["k"], case.get("count", 1)
        if case.get("prec", "plain") != "plain":
            a, b = _wide(g, m * k), _wide(g, k * n)
        else:
            t = {"half": HALF, "complex": CPLX}.get(kind, REAL)[dtype]
            a, b = _uniform(g, m * k * count, t), _uniform(g, k * n * count, t)
        c = torch.float32 if kind == "half" else (CPLX if kind == "complex" else REAL)[dtype]
        return a, b, _uniform(g, m * n * count, c)
    if kind == "gemv":
        t = (CPLX if case["field"] == "complex" else REAL)[dtype]
        x, y = (n, m) if case["op"] == "N" else (m, n)
        return _uniform(g, m * n, t), _uniform(g, x, t), _uniform(g, y, t)
    t = REAL[dtype]
    if kind == "level3" and case["routine"] == "syrk":  # C (m x m) from A with inner dimension n
        return _uniform(g, m * n, t), None, _uniform(g, m * m, t)
    order = m if case["side"] == "L" else n
    a = _triangle(g, order, t)
    return a, _uniform(g, m * n, t), _uniform(g, m * n, t)


def _problems(case, data):
    """The batch's product descriptors: C_p = A_p * B_p."""
    dims, half, out = _batch_shapes(case).tolist(), case["count"] // 2, []
    for name, part in (("f32", dims[:half]), ("f64", dims[half:])):
        size = data[name][0].element_size()
        pa, pb, pc = (t.data_ptr() for t in data[name])
        for m, n, k in part:
            out.append(E.GemmProblem(dtype=CODE[name], opa=0, opb=0, reserved=0, m=m, n=n, k=k, lda=m, ldb=k, ldc=m,
                                     A=ctypes.c_void_p(pa), B=ctypes.c_void_p(pb), C=ctypes.c_void_p(pc), alpha=1.0,
                                     beta=0.0))
            pa, pb, pc = pa + m * k * size, pb + k * n * size, pc + m * n * size
    return out


def prepare(case, seed):
    data = _inputs(case, seed)
    state = dict(case=case, data=data)
    if case["kind"] == "grouped":
        state["batch"] = E.Grouped(_problems(case, data))
    elif case["kind"] == "trsm" or case.get("routine") == "trmm":
        state["x"] = torch.empty_like(data[1])
    return state


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "grouped":
        state["batch"].graph_launch()
        return {name: state["data"][name][2] for name in ("f32", "f64")}
    a, b, c = state["data"]
    m, n = case["m"], case["n"]
    if kind == "gemm":
        k = case["k"]
        E.gemm(CODE[case["dtype"]], OPS[case["opa"]], OPS[case["opb"]], m, n, k, case["alpha"], a,
               _stored(case["opa"], m, k)[0], b, _stored(case["opb"], k, n)[0], case["beta"], c, m,
               prec=PRECS[case["prec"]])
        return c
    if kind == "half":
        k = case["k"]
        f = E.gemm_bf16 if case["dtype"] == "bf16" else E.gemm_f16
        f(OPS[case["opa"]], OPS[case["opb"]], m, n, k, case["alpha"], a, _stored(case["opa"], m, k)[0], b,
          _stored(case["opb"], k, n)[0], case["beta"], c, m)
        return c
    if kind == "complex":
        k = case["k"]
        E.gemm_complex(CODE[case["dtype"]], OPS[case["opa"]], OPS[case["opb"]], m, n, k, 1.0 + 0.5j, a,
                       _stored(case["opa"], m, k)[0], b, _stored(case["opb"], k, n)[0], 0.5, c, m, prec=E.PREC_PLAIN)
        return c
    if kind == "gemv":
        f = E.gemv_complex if case["field"] == "complex" else E.gemv
        f(CODE[case["dtype"]], OPS[case["op"]], m, n, 1.0, a, m, b, 1, 0.0, c, 1)
        return c
    if kind == "strided":
        k = case["k"]
        E.gemm_batched_strided(CODE[case["dtype"]], OPS[case["opa"]], OPS[case["opb"]], m, n, k, 1.0, a,
                               _stored(case["opa"], m, k)[0], m * k, b, _stored(case["opb"], k, n)[0], k * n, 0.0, c,
                               m, m * n, case["count"])
        return c
    uplo, side = (E.LOWER if case["uplo"] == "L" else E.UPPER), (E.LEFT if case["side"] == "L" else E.RIGHT)
    dt, op, order = CODE[case["dtype"]], OPS[case["op"]], m if case["side"] == "L" else n
    if kind == "trsm" or case["routine"] == "trmm":  # in place: the right-hand sides are kept, so copied first
        x = state["x"]
        x.copy_(b)
        f = E.trsm if kind == "trsm" else E.trmm
        f(dt, side, uplo, op, E.NON_UNIT, m, n, 1.0, a, order, x, m)
        return x
    if case["routine"] == "symm":
        E.symm(dt, side, uplo, m, n, 1.0, a, order, b, m, 0.5, c, m)
    else:
        E.syrk(dt, uplo, op, m, n, 1.0, a, _stored(case["op"], m, n)[0], 0.5, c, m)
    return c


def work(case):
    kind = case["kind"]
    if kind == "grouped":
        dims, half = _batch_shapes(case).astype(float), case["count"] // 2
        m, n, k = dims.T
        size = np.where(np.arange(len(dims)) < half, 4, 8)
        return {"bytes": float(((m * k + k * n + m * n) * size).sum()), "flops": float((2 * m * n * k).sum())}
    m, n, size = case["m"], case["n"], {"f32": 4, "f64": 8, "bf16": 2, "f16": 2}[case["dtype"]]
    if kind in ("gemm", "half", "complex", "strided"):
        k, count, c = case["k"], case.get("count", 1), 2 if kind == "complex" else 1
        reads = 2 if kind == "complex" or case.get("beta", 0.0) != 0.0 else 1
        out = 4 if kind == "half" else size * c
        return {"bytes": float(count * ((m * k + k * n) * size * c + m * n * out * reads)),
                "flops": 2.0 * c * c * m * n * k * count}
    if kind == "gemv":
        c = 2 if case["field"] == "complex" else 1
        return {"bytes": float((m * n + m + n) * size * c), "flops": 2.0 * c * c * m * n}
    if case.get("routine") == "syrk":
        return {"bytes": float((m * n + m * (m + 1)) * size), "flops": float(m) * m * n}
    order = m if case["side"] == "L" else n
    if case.get("routine") == "symm":
        return {"bytes": float((order * (order + 1) // 2 + 3 * m * n) * size), "flops": 2.0 * order * m * n}
    return {"bytes": float((order * (order + 1) // 2 + 2 * m * n) * size), "flops": float(order) * m * n}


# ---- 64-bit reference ---------------------------------------------------------------

def _wide_type(t):
    return t.to(torch.complex128 if t.is_complex() else torch.float64)


def _mat(flat, op, rows, cols):
    """op() of a stored flat column-major matrix, as a rows x cols torch matrix."""
    r, c = _stored(op, rows, cols)
    x = _wide_type(flat).view(c, r).T
    return x if op == "N" else (x.T if op == "T" else x.conj().T)


def _flat(x):
    return x.T.contiguous().reshape(-1)


def exact(case, seed):
    data, kind = _inputs(case, seed), case["kind"]
    if kind == "grouped":
        dims, half, out = _batch_shapes(case).tolist(), case["count"] // 2, {}
        for name, part in (("f32", dims[:half]), ("f64", dims[half:])):
            a, b, c = (t.double() for t in data[name])
            pa = pb = pc = 0
            for m, n, k in part:  # C^T = B^T A^T, stored rows of the transposes
                torch.matmul(b[pb:pb + k * n].view(n, k), a[pa:pa + m * k].view(k, m), out=c[pc:pc + m * n].view(n, m))
                pa, pb, pc = pa + m * k, pb + k * n, pc + m * n
            out[name] = c
        return out
    a, b, c = data
    m, n = case["m"], case["n"]
    if kind in ("gemm", "half"):
        k = case["k"]
        r = case["alpha"] * (_mat(a, case["opa"], m, k) @ _mat(b, case["opb"], k, n))
        return _flat(r if case["beta"] == 0.0 else r + case["beta"] * _mat(c, "N", m, n))
    if kind == "complex":
        k = case["k"]
        r = _mat(a, case["opa"], m, k).resolve_conj().contiguous() @ _mat(b, case["opb"], k, n).resolve_conj().contiguous()
        return _flat((1.0 + 0.5j) * r + 0.5 * _mat(c, "N", m, n))
    if kind == "gemv":
        x = _wide_type(a).view(n, m)
        return (x.T if case["op"] == "N" else x) @ _wide_type(b)
    if kind == "strided":
        k, count = case["k"], case["count"]
        (ra, ca), (rb, cb) = _stored(case["opa"], m, k), _stored(case["opb"], k, n)
        at, bt = a.double().view(count, ca, ra), b.double().view(count, cb, rb)  # the stored transposes
        at = at if case["opa"] == "N" else at.transpose(1, 2).contiguous()
        bt = bt if case["opb"] == "N" else bt.transpose(1, 2).contiguous()
        return torch.bmm(bt, at).reshape(-1)
    if case.get("routine") == "syrk":
        x = _mat(a, case["op"], m, n)
        old = _mat(c, "N", m, m)
        new = x @ x.T + 0.5 * old
        keep = torch.ones(m, m, dtype=torch.bool, device=DEV)
        return _flat(torch.where(keep.tril() if case["uplo"] == "L" else keep.triu(), new, old))
    order = m if case["side"] == "L" else n
    s = a.double().view(order, order).T
    t = s.tril() if case["uplo"] == "L" else s.triu()
    x = _mat(b, "N", m, n)
    if case.get("routine") == "symm":
        full = t + (t.tril(-1) if case["uplo"] == "L" else t.triu(1)).T
        return _flat((full @ x if case["side"] == "L" else x @ full) + 0.5 * _mat(c, "N", m, n))
    t = t if case["op"] == "N" else t.T
    if case.get("routine") == "trmm":
        return _flat(t @ x if case["side"] == "L" else x @ t)
    lower = (case["uplo"] == "L") == (case["op"] == "N")
    return _flat(torch.linalg.solve_triangular(t.contiguous(), x.contiguous(), upper=not lower,
                                               left=case["side"] == "L"))
