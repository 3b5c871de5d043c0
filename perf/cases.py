"""The measured workloads of the library: one pass each through its public C API.

Every case calls the entry points of clgpu_amd.iclblas (or, for the training step,
the autograd functions built on them) on device-resident column-major matrices, the
way a GPU program holds them. A rows x cols matrix of leading dimension ld is a torch
tensor of shape (cols, ld). Host-pointer calls run the same kernels between two PCIe
copies and are not measured here.

The sizes are the library's own configurations (SGEMM 256^3 and 8192^3, CGEMM 4096^3,
STRSM 4096 x 1024, the 2048 chain, SGEMV 16384^2) and, around them, sizes as they come
in use: ragged, with odd leading dimensions, all ops, sides and triangles.
"""
import math

import torch

from clgpu_amd import autograd
from clgpu_amd import iclblas as ib

LARGEST = 2.0 * 8192 ** 3  # flops of the largest listed case


def listed():
    """The cases; "op" names the routine, the other keys its arguments."""
    return [
        # The smallest call: one 256^3 update C = A B + C / 2, where launch latency counts.
        dict(name="sgemm_256", op="gemm", cplx=False, split=False, ta=0, tb=0, m=256, n=256, k=256,
             pa=0, pb=0, pc=0, alpha=1.0, beta=0.5),
        # An ordinary product of data whose sizes nobody rounded: odd everywhere, so no
        # column but the first is 16-byte aligned (activations x weights^T).
        dict(name="sgemm_ragged", op="gemm", cplx=False, split=False, ta=0, tb=1, m=1111, n=2003, k=1777,
             pa=0, pb=0, pc=2, alpha=1.0, beta=0.0),
        # The headline product on the FP32 path.
        dict(name="sgemm_8192", op="gemm", cplx=False, split=False, ta=0, tb=0, m=8192, n=8192, k=8192,
             pa=0, pb=0, pc=0, alpha=1.0, beta=0.0),
        # The headline product in the split-BF16 math mode.
        dict(name="sgemm_8192_split", op="gemm", cplx=False, split=True, ta=0, tb=0, m=8192, n=8192, k=8192,
             pa=0, pb=0, pc=0, alpha=1.0, beta=0.0),
        # Complex product with a conjugate-transposed operand, complex alpha and beta (beamforming).
        dict(name="cgemm_4096_cn", op="gemm", cplx=True, split=False, ta=2, tb=0, m=4096, n=4096, k=4096,
             pa=0, pb=0, pc=0, alpha=1.0, alpha_im=0.5, beta=0.25),
        # Triangular solve, many right-hand sides (the solve of a factored system).
        dict(name="strsm_4096", op="trsm", cplx=False, side=0, uplo=1, trans=0, diag=0, m=4096, n=1024, pa=0, pb=0),
        # Complex solve from the right with the conjugate transpose of an upper triangle, ragged
        # (a whitening step with a Cholesky factor).
        dict(name="ctrsm_ragged", op="trsm", cplx=True, side=1, uplo=0, trans=2, diag=0, m=701, n=1153, pa=2, pb=0),
        # Gram matrix A^T A of tall data: a small triangle, a long sum.
        dict(name="ssyrk_gram", op="syrk", cplx=False, uplo=1, trans=1, n=640, k=20011, pa=0, pc=0),
        # Product with a triangular factor.
        dict(name="strmm_3000", op="trmm", cplx=False, side=0, uplo=1, trans=0, diag=0, m=3000, n=2000, pa=0, pb=0, pc=0),
        # Matrix-vector product, HBM-bound: the largest, and a ragged one of ordinary size.
        dict(name="sgemv_16384", op="gemv", cplx=False, trans=0, m=16384, n=16384, pa=0, incx=1, incy=1),
        dict(name="sgemv_ragged_t", op="gemv", cplx=False, trans=1, m=3001, n=2003, pa=0, incx=1, incy=1),
        # A training step: forward and backward of X = A^-1 (alpha G H), loss = sum(W * X).
        dict(name="chain_2048", op="chain", order=2048, lines=512, alpha=0.5),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]; half of them rounded to a multiple of 64."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return max(lo, v // 64 * 64) if v >= 128 and rng.random() < 0.5 else v


def draw(rng):
    """One more case: any routine of the listed ones, any op, side and triangle, sizes over the whole range."""
    while True:
        case = _draw_one(rng)
        if 1e5 < work(case)["flops"] <= LARGEST:
            return case


def _draw_one(rng):
    op = rng.choice(["gemm", "gemm", "gemm", "trsm", "syrk", "trmm", "gemv", "chain"])
    cplx = op != "chain" and rng.random() < 0.35
    pad = lambda: rng.choice([0, 0, 0, 1, 3, 64])  # noqa: E731
    trans = rng.choice([0, 1, 2] if cplx else [0, 1])
    if op == "gemm":
        case = dict(op=op, cplx=cplx, split=rng.random() < 0.3, ta=trans, tb=rng.choice([0, 1, 2] if cplx else [0, 1]),
                    m=_log(rng, 64, 8192), n=_log(rng, 64, 8192), k=_log(rng, 64, 8192), pa=pad(), pb=pad(), pc=pad(),
                    alpha=rng.choice([1.0, -0.5]), beta=rng.choice([0.0, 0.0, 0.5]))
        if cplx:
            case["alpha_im"] = rng.choice([0.0, 0.5])
        return case
    if op == "trsm":
        return dict(op=op, cplx=cplx, side=rng.choice([0, 1]), uplo=rng.choice([0, 1]), trans=trans,
                    diag=rng.choice([0, 0, 1]), m=_log(rng, 64, 4096), n=_log(rng, 64, 4096), pa=pad(), pb=pad())
    if op == "syrk":
        return dict(op=op, cplx=cplx, uplo=rng.choice([0, 1]), trans=trans, n=_log(rng, 64, 6000),
                    k=_log(rng, 64, 24000), pa=pad(), pc=pad())
    if op == "trmm":
        return dict(op=op, cplx=cplx, side=rng.choice([0, 1]), uplo=rng.choice([0, 1]), trans=trans,
                    diag=rng.choice([0, 0, 1]), m=_log(rng, 64, 6000), n=_log(rng, 64, 6000), pa=pad(), pb=pad(), pc=pad())
    if op == "gemv":
        return dict(op=op, cplx=cplx, trans=trans, m=_log(rng, 256, 16384), n=_log(rng, 256, 16384), pa=pad(),
                    incx=rng.choice([1, 1, 2]), incy=rng.choice([1, 1, 2]))
    return dict(op=op, order=_log(rng, 128, 3000), lines=_log(rng, 64, 1024), alpha=0.5)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
_handles = {}


def _handle(split):
    """The program's handles: device pointers, torch's stream, one per math mode, kept for its life."""
    if split not in _handles:
        _handles[split] = ib.Handle(memory_mode=ib.MEMORY_DEVICE,
                                    math_mode=ib.MATH_SPLIT_BF16X3 if split else ib.MATH_FP32,
                                    stream=torch.cuda.current_stream().cuda_stream)
    return _handles[split]


def _matrix(gen, rows, cols, pad, cplx):
    """Column-major rows x cols matrix, entries uniform in [-1, 1] (both parts of a complex one)."""
    shape = (cols, rows + pad) + ((2,) if cplx else ())
    t = torch.empty(shape, device="cuda", dtype=torch.float32).uniform_(-1.0, 1.0, generator=gen)
    return torch.view_as_complex(t) if cplx else t


def _triangular(gen, order, pad, cplx):
    """A well-conditioned triangular factor: diagonal +-[1, 2], the rest uniform / sqrt(order)."""
    t = _matrix(gen, order, order, pad, cplx) / math.sqrt(order)
    d = torch.empty(order, device="cuda").uniform_(1.0, 2.0, generator=gen)
    sign = torch.randint(0, 2, (order,), device="cuda", generator=gen) * 2 - 1
    t[:, :order].diagonal().copy_(d * sign)
    return t


def _shapes(case):
    """(rows, cols) of the stored operands."""
    op = case["op"]
    if op == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return ((m, k) if case["ta"] == 0 else (k, m)), ((k, n) if case["tb"] == 0 else (n, k))
    if op == "syrk":
        return ((case["n"], case["k"]) if case["trans"] == 0 else (case["k"], case["n"])), None
    return None, None


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    op, s = case["op"], dict(case=case)
    if op == "chain":
        o, lines = case["order"], case["lines"]
        s["A"] = _triangular(gen, o, 0, False).requires_grad_()
        s["G"] = _matrix(gen, o, o, 0, False).requires_grad_()
        s["H"] = _matrix(gen, o, lines, 0, False).requires_grad_()
        s["W"] = torch.randn((lines, o), device="cuda", generator=gen)
        return s
    cplx = case["cplx"]
    s["h"] = _handle(case.get("split", False))
    if op == "gemm":
        (ra, ca), (rb, cb) = _shapes(case)
        s["A"] = _matrix(gen, ra, ca, case["pa"], cplx)
        s["B"] = _matrix(gen, rb, cb, case["pb"], cplx)
        s["C"] = _matrix(gen, case["m"], case["n"], case["pc"], cplx)
    elif op == "trsm":
        s["A"] = _triangular(gen, case["m"] if case["side"] == 0 else case["n"], case["pa"], cplx)
        s["B"] = _matrix(gen, case["m"], case["n"], case["pb"], cplx)
        s["X"] = torch.empty_like(s["B"])
    elif op == "syrk":
        (ra, ca), _ = _shapes(case)
        s["A"] = _matrix(gen, ra, ca, case["pa"], cplx)
        s["C"] = _matrix(gen, case["n"], case["n"], case["pc"], cplx)
    elif op == "trmm":
        s["A"] = _triangular(gen, case["m"] if case["side"] == 0 else case["n"], case["pa"], cplx)
        s["B"] = _matrix(gen, case["m"], case["n"], case["pb"], cplx)
        s["C"] = _matrix(gen, case["m"], case["n"], case["pc"], cplx)
    else:  # gemv
        m, n = case["m"], case["n"]
        lenx, leny = (n, m) if case["trans"] == 0 else (m, n)
        s["A"] = _matrix(gen, m, n, case["pa"], cplx)
        s["x"] = _matrix(gen, lenx * case["incx"], 1, 0, cplx)[0]
        s["y"] = _matrix(gen, leny * case["incy"], 1, 0, cplx)[0]
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def _scalars(case):
    alpha, beta = case.get("alpha", 1.0), case.get("beta", 0.0)
    return (complex(alpha, case.get("alpha_im", 0.0)), complex(beta, 0.0)) if case["cplx"] else (alpha, beta)


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "chain":
        X = autograd.strsm(state["A"], autograd.sgemm(state["G"], state["H"], case["alpha"]))
        loss = (state["W"] * X).sum()
        dA, dG, dH = torch.autograd.grad(loss, [state["A"], state["G"], state["H"]])
        return dict(X=X, dA=dA, dG=dG, dH=dH)
    h, cplx, A = state["h"].value, case["cplx"], state["A"]
    lda = A.shape[1]
    if op == "gemm":
        alpha, beta = _scalars(case)
        B, C = state["B"], state["C"]
        call = ib.iclblasCgemm if cplx else ib.iclblasSgemm
        ib.check(call(h, case["ta"], case["tb"], case["m"], case["n"], case["k"], alpha, A, lda, B, B.shape[1], beta,
                      C, C.shape[1]), "gemm")
        return C
    if op == "trsm":  # solves in place: the right-hand side is kept and copied first
        X = state["X"].copy_(state["B"])
        call = ib.iclblasCtrsm if cplx else ib.iclblasStrsm
        ib.check(call(h, case["side"], case["uplo"], case["trans"], case["diag"], case["m"], case["n"], 1.0, A, lda,
                      X, X.shape[1]), "trsm")
        return X
    if op == "syrk":
        C = state["C"]
        call = ib.iclblasCsyrk if cplx else ib.iclblasSsyrk
        ib.check(call(h, case["uplo"], case["trans"], case["n"], case["k"], 1.0, A, lda, 0.0, C, C.shape[1]), "syrk")
        return C
    if op == "trmm":
        B, C = state["B"], state["C"]
        call = ib.iclblasCtrmm if cplx else ib.iclblasStrmm
        ib.check(call(h, case["side"], case["uplo"], case["trans"], case["diag"], case["m"], case["n"], 1.0, A, lda,
                      B, B.shape[1], C, C.shape[1]), "trmm")
        return C
    x, y = state["x"], state["y"]
    call = ib.iclblasCgemv if cplx else ib.iclblasSgemv
    ib.check(call(h, case["trans"], case["m"], case["n"], 1.0, A, lda, x, case["incx"], 0.0, y, case["incy"]), "gemv")
    return y


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    op = case["op"]
    if op == "chain":
        o, r = float(case["order"]), float(case["lines"])
        # forward: G H and the solve; backward: the solve, dA = -tri(dB X^T), dG, dH
        flops = 2 * o * o * r + o * o * r + o * o * r + o * o * r + 2 * (2 * o * o * r)
        # inputs A (a triangle), G, H, W; outputs X, dA, dG, dH
        return {"bytes": 4 * (0.5 * o * o + o * o + 2 * o * r + o * r + 2 * o * o + o * r), "flops": flops}
    c = 4.0 if case["cplx"] else 1.0  # real multiply-adds per element's
    es = 8.0 if case["cplx"] else 4.0
    if op == "gemm":
        m, n, k = float(case["m"]), float(case["n"]), float(case["k"])
        reads_c = 1.0 if case["beta"] else 0.0
        return {"bytes": es * (m * k + k * n + (1 + reads_c) * m * n), "flops": c * 2 * m * n * k}
    if op == "syrk":
        n, k = float(case["n"]), float(case["k"])
        return {"bytes": es * (n * k + n * n / 2), "flops": c * n * n * k}
    m, n = float(case["m"]), float(case["n"])
    if op == "gemv":
        return {"bytes": es * (m * n + m + n), "flops": c * 2 * m * n}
    order, lines = (m, n) if case["side"] == 0 else (n, m)
    return {"bytes": es * (order * order / 2 + 2 * m * n), "flops": c * order * order * lines}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _mat(t, rows):
    """The rows x cols matrix a column-major tensor holds, in 64 bits."""
    return t[:, :rows].t().to(torch.complex128 if t.is_complex() else torch.float64)


def _op(M, trans):
    return M if trans == 0 else M.t() if trans == 1 else M.conj().t()


def _mm(P, Q):
    return P.resolve_conj().contiguous() @ Q.resolve_conj().contiguous()


def _stored(old, M):
    """`old` in 64 bits with the matrix M written over its leading rows."""
    out = old.to(torch.complex128 if old.is_complex() else torch.float64)
    out[:, :M.shape[0]] = M.t()
    return out


def _tri_op(case, s, order):
    """(op(A) with the other triangle and, for a unit diagonal, the diagonal set, op(A) is upper)."""
    T = _mat(s["A"], order)
    T = T.tril() if case["uplo"] == 1 else T.triu()
    if case["diag"] == 1:
        T.diagonal().fill_(1.0)
    return _op(T, case["trans"]).resolve_conj().contiguous(), (case["uplo"] == 0) == (case["trans"] == 0)


def exact(case, seed):
    s, op = prepare(case, seed), case["op"]
    if op == "chain":
        o, alpha = case["order"], case["alpha"]
        T = _mat(s["A"].detach(), o).tril()
        G, H, W = _mat(s["G"].detach(), o), _mat(s["H"].detach(), o), _mat(s["W"], o)
        X = torch.linalg.solve_triangular(T, alpha * _mm(G, H), upper=False)
        dB = torch.linalg.solve_triangular(T.t().contiguous(), W.contiguous(), upper=True)
        cm = lambda M: M.t().contiguous()  # noqa: E731
        return dict(X=cm(X), dA=cm(-_mm(dB, X.t()).tril()), dG=cm(alpha * _mm(dB, H.t())), dH=cm(alpha * _mm(G.t(), dB)))
    if op == "gemm":
        alpha, beta = _scalars(case)
        (ra, _), (rb, _) = _shapes(case)
        P = _mm(_op(_mat(s["A"], ra), case["ta"]), _op(_mat(s["B"], rb), case["tb"]))
        P = alpha * P
        if beta:
            P = P + beta * _mat(s["C"], case["m"])
        return _stored(s["C"], P)
    if op == "syrk":
        n = case["n"]
        (ra, _), _ = _shapes(case)
        O = _op(_mat(s["A"], ra), case["trans"])
        P, old = _mm(O, O.t()), _mat(s["C"], n)
        P = P.tril() + old.triu(1) if case["uplo"] == 1 else P.triu() + old.tril(-1)
        return _stored(s["C"], P)
    if op in ("trsm", "trmm"):
        left = case["side"] == 0
        order = case["m"] if left else case["n"]
        T, upper = _tri_op(case, s, order)
        B = _mat(s["B"], case["m"]).contiguous()
        if op == "trmm":
            return _stored(s["C"], _mm(T, B) if left else _mm(B, T))
        return _stored(s["B"], torch.linalg.solve_triangular(T, B, upper=upper, left=left))
    m, n, x, y = case["m"], case["n"], s["x"], s["y"]
    wide = torch.complex128 if case["cplx"] else torch.float64
    out = y.to(wide)
    A = _op(_mat(s["A"], m), case["trans"]).resolve_conj()
    out[::case["incy"]] = A @ x[::case["incx"]].to(wide)
    return out
