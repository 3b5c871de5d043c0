"""The range guard of the three-way split kernels on every path that it has to stop (the triangle's two
launches, windows of a triangular operand, parts of a split depth) and every kernel that runs behind it,
and operands at the ends of the range."""
import pytest

from blas_helpers import U32
from clgpu_amd import iclblas as ib

pytestmark = pytest.mark.gpu
REAL = [n for n in ib.implementation_names() if n.startswith("sgemm_f32_split3")]
CPLX = [n for n in ib.implementation_names() if n.startswith("cgemm_f32_split3")]
ALPHA, BETA = 0.75, -0.5


def _call(h, op, uplo, m, n, k, A, B, C):
    """C = ALPHA op + BETA C in place; device tensors are column major (torch's rows are columns)."""
    p = [t if t is None else t.data_ptr() for t in (A, B, C)]
    if op == "gemm":
        return ib.iclblasSgemm(h.value, 0, 0, m, n, k, ALPHA, p[0], m, p[1], k, BETA, p[2], m)
    if op == "syrk":
        return ib.iclblasSsyrk(h.value, uplo, 0, n, k, ALPHA, p[0], n, BETA, p[2], n)
    if op == "herk":
        return ib.iclblasCherk(h.value, uplo, 0, n, k, ALPHA, p[0], n, BETA, p[2], n)
    trmm = ib.iclblasCtrmm if A.is_complex() else ib.iclblasStrmm
    return trmm(h.value, 0, uplo, 0, 0, m, n, ALPHA, p[0], m, p[1], m, p[2], m)


def _exact(op, uplo, A, B, C):
    """(result, magnitude, written) as matrices of torch's rows, in float64."""
    import torch
    wide = torch.complex128 if C.is_complex() else torch.float64
    A, C = A.to(wide), C.to(wide)
    tri = (lambda X: X.tril()) if uplo == 0 else (lambda X: X.triu())  # rows are columns: upper is tril
    ones = torch.ones(C.shape, device=C.device, dtype=torch.bool)
    if op == "gemm":
        B = B.to(wide)
        return ALPHA * B @ A + BETA * C, ALPHA * B.abs() @ A.abs() + abs(BETA) * C.abs(), ones
    if op in ("syrk", "herk"):
        X = (A.conj() if op == "herk" else A).T.contiguous()
        E, mag = ALPHA * X @ A + BETA * C, ALPHA * X.abs() @ A.abs() + abs(BETA) * C.abs()
        if op == "herk":
            E.diagonal().imag.zero_()
        return E, mag, tri(ones)
    A, B = tri(A), B.to(wide)
    return ALPHA * B @ A, ALPHA * B.abs() @ A.abs(), ones


CASES = [("syrk", 0, None, 1027, 300), ("syrk", 1, None, 640, 4100), ("herk", 1, None, 700, 130), ("herk", 0, None, 300, 2100),
         ("trmm", 1, 700, 300, 700), ("trmm", 0, 520, 260, 520), ("ctrmm", 1, 400, 300, 400), ("gemm", 0, 128, 128, 20011),
         ("gemm", 0, 700, 900, 3000), ("gemm", 0, 2048, 2048, 512)]


@pytest.mark.parametrize("tile", [0, 1])
@pytest.mark.parametrize("op,uplo,m,n,k", CASES)
def test_guarded_paths(dev_handle, op, uplo, m, n, k, tile):
    """One element outside the range, then many, then none: always the product, applied once, and the same
    result with the operand back in range."""
    import torch
    h = dev_handle
    cplx = op in ("herk", "ctrmm")
    impl = (CPLX if cplx else REAL)[tile]
    op = "trmm" if op == "ctrmm" else op
    gen = torch.Generator("cuda").manual_seed(21)
    rnd = lambda r, c: torch.rand((r, c), device="cuda", generator=gen,  # noqa: E731
                                  dtype=torch.complex64 if cplx else torch.float32) - (0.5 + 0.5j if cplx else 0.5)
    A = rnd(k, n if op in ("syrk", "herk") else m)
    B = None if op in ("syrk", "herk") else rnd(n, k)
    C0 = rnd(n, n if op in ("syrk", "herk") else m)
    if op == "herk":
        C0.diagonal().imag.zero_()
    A0 = A.clone()
    h.set_math_mode(ib.MATH_FP32)
    h.set_implementation(impl)
    clean = None
    try:
        for outside in ("none", "one", "none", "many", "none"):
            A.copy_(A0)
            if outside == "one":
                A[k // 3, A.shape[1] // 3 if uplo == 0 else A.shape[1] - 1] = 2.0 ** 50
            elif outside == "many":
                A[torch.rand(A.shape, device="cuda", generator=gen) < 0.01] = 2.0 ** -115
            C = C0.clone()
            torch.cuda.synchronize()
            ib.check(_call(h, op, uplo, m, n, k, A, B, C))
            h.synchronize()
            assert h.last_implementation() == impl
            E, mag, written = _exact(op, uplo, A, B, C0)
            kk = 2 * k if cplx else k
            assert bool(((C - E).abs() <= 4 * (kk + 2) * U32 * (2 if cplx else 1) * mag)[written].all())
            assert torch.equal(C[~written], C0[~written])
            if outside == "none":
                clean = C if clean is None else clean
                assert torch.equal(C, clean)
    finally:
        h.set_implementation(None)


@pytest.mark.parametrize("impl", REAL)
@pytest.mark.parametrize("lo,hi,blo,bhi", [(49, 50, 49, 50), (-110, -109, 49, 50), (-110, -60, 0, 1), (-70, -50, -70, -50),
                                           (-66, -60, -66, -60), (-110, -60, -60, -30)])
def test_ends_of_the_range(dev_handle, impl, lo, hi, blo, bhi):
    """Operands of magnitudes 2^lo to 2^hi and 2^blo to 2^bhi. Where products fall below the normal range,
    each of the six partial ones may be cut off at the smallest subnormal number."""
    import torch
    m, n, k = 260, 130, 300
    gen = torch.Generator("cuda").manual_seed(22)

    def rnd(r, c, lo, hi):
        x = torch.rand((r, c), device="cuda", generator=gen, dtype=torch.float64)
        s = torch.rand((r, c), device="cuda", generator=gen) - 0.5
        x = (torch.exp2(lo + (hi - lo) * x).float().clamp(2.0 ** lo, 2.0 ** hi * (1 - 2.0 ** -24)) * s.sign())
        x[0, 0], x[1, 1] = 2.0 ** lo, 2.0 ** hi * (1 - 2.0 ** -24)
        return x
    A, B = rnd(k, m, lo, hi), rnd(n, k, blo, bhi)
    C = torch.zeros((n, m), device="cuda")
    h = dev_handle
    h.set_math_mode(ib.MATH_FP32)
    h.set_implementation(impl)
    torch.cuda.synchronize()
    try:
        ib.check(ib.iclblasSgemm(h.value, 0, 0, m, n, k, 1.0, A, m, B, k, 0.0, C, m))
        h.synchronize()
        assert h.last_implementation() == impl
    finally:
        h.set_implementation(None)
    X, Y = A.double(), B.double()
    bound = 4 * k * U32 * (Y.abs() @ X.abs()) + 6 * k * 2.0 ** -149
    assert bool(((C.double() - Y @ X).abs() <= bound).all())
