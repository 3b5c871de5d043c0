"""The 32 x 32 tile kernels whose waves share the depth (*gemm_f32_wave_32x32): edges of the
tile, of a wave's block of the depth (32, complex 8) and of the eight waves' round (256, 64)
against the FP64 oracle, and the level-3 options."""
import numpy as np
import pytest

import oracle
from blas_helpers import U32, bound_ratio
from clgpu_amd import datagen
from clgpu_amd import iclblas as ib
from l3_helpers import RANK2K, RANKK, call_library, oracle_result, random_case, shapes

pytestmark = pytest.mark.gpu
SHAPES = [(1, 1, 1), (2, 3, 7), (33, 31, 8), (32, 32, 32), (31, 65, 33), (64, 1, 64), (65, 66, 257), (100, 40, 520)]


@pytest.fixture
def h(handle):
    handle.set_math_mode(ib.MATH_FP32)
    yield handle
    handle.set_implementation(None)


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("ta", [0, 1, 2])
@pytest.mark.parametrize("tb", [0, 1, 2])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_edges(h, cplx, ta, tb, shape):
    m, n, k = shape
    ra, ca = (m, k) if ta == 0 else (k, m)
    rb, cb = (k, n) if tb == 0 else (n, k)
    mat = datagen.complex_matrix if cplx else datagen.matrix
    A, B, C = mat(ra, ca, ra + 3, "A", seed=43), mat(rb, cb, rb + 1, "B", seed=43), mat(m, n, m + 2, "C", seed=43)
    A[ra:], B[rb:] = np.nan, np.nan  # padding rows are never used
    C0 = C.copy(order="F")
    alpha, beta = (0.5 - 1.5j, 0.25 + 1.0j) if cplx else (-1.5, 0.5)
    f64 = oracle.zgemm if cplx else oracle.dgemm
    E, ab = f64(ta, tb, m, n, k, alpha, A, B, beta, C)
    impl = ("c" if cplx else "s") + "gemm_f32_wave_32x32"
    h.set_implementation(impl)
    f = ib.iclblasCgemm if cplx else ib.iclblasSgemm
    ib.check(f(h.value, ta, tb, m, n, k, alpha, A, ra + 3, B, rb + 1, beta, C, m + 2))
    assert h.last_implementation() == impl
    c = 2 if cplx else 1
    wide = np.complex128 if cplx else np.float64
    extra = 2 * c * U32 * (abs(beta) * np.abs(C0[:m].astype(wide)) + abs(alpha) * ab)
    assert bound_ratio(np.abs(C[:m].astype(wide) - E), c * k, abs(alpha) * ab, extra) <= 4.0
    assert np.array_equal(C[m:], C0[m:])


LEVEL3 = [("Ssyrk", dict(uplo=1, trans=1), (None, 70, 33)), ("Ssyrk", dict(uplo=0, trans=0), (None, 129, 260)),
          ("Ssyr2k", dict(uplo=1, trans=0), (None, 67, 40)), ("Cherk", dict(uplo=0, trans=2), (None, 65, 70)),
          ("Csyrk", dict(uplo=1, trans=0), (None, 96, 9)), ("Cher2k", dict(uplo=1, trans=0), (None, 66, 20)),
          ("Ssymm", dict(side=1, uplo=0), (33, 75, None)), ("Chemm", dict(side=0, uplo=1), (70, 34, None))] + [
    (r, dict(side=s, uplo=u, trans=t, diag=d), (97, 40, None) if s == 0 else (40, 97, None))
    for r in ("Strmm", "Ctrmm") for s in (0, 1) for u in (0, 1) for t, d in ((0, 0), (2, 1))]


@pytest.mark.parametrize("routine,v,shape", LEVEL3, ids=lambda x: str(x).replace(" ", ""))
def test_level3_options(h, routine, v, shape):
    m, n, k = shape
    c = random_case(routine, np.random.default_rng(n), m=m, n=n, k=k, **v)
    impl = routine[0].lower() + "gemm_f32_wave_32x32"
    h.set_implementation(impl)
    A, B, C = c["A"].copy(order="F"), (c["B"].copy(order="F") if c.get("B") is not None else None), c["C"].copy(order="F")
    ib.check(call_library(h.value, c, A, B, C), routine)
    assert h.last_implementation() == impl
    exp, mag, kk = oracle_result(c, c["A"], c.get("B"), c["C"])
    (rc, cc) = shapes(c)[2]
    written = np.ones((rc, cc), bool)
    if routine in RANKK or routine in RANK2K:
        written = np.tril(written) if v["uplo"] == 1 else np.triu(written)
    C0 = np.abs(np.nan_to_num(c["C"][:rc, :cc].astype(np.complex128)))
    bound = 4.0 * (kk + 2) * U32 * (abs(c["alpha"]) * mag + abs(c.get("beta", 0.0)) * C0)
    err = np.abs(C[:rc, :cc].astype(np.complex128) - exp[:rc, :cc])
    assert np.all((err <= bound + 1e-30)[written])
    assert np.array_equal(C[:rc, :cc][~written], c["C"][:rc, :cc][~written])
    assert np.array_equal(C[rc:], c["C"][rc:])
