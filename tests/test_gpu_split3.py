"""FP32 products on the three-way split kernels (*gemm_f32_split3_*): edges of the
tiles and of the 32-deep slabs against the FP64 oracle, the level-3 options, the
range guard (operands the split does not cover give the FP32 MFMA result bit for
bit), and the calls that must stay off the optional workspace."""
import numpy as np
import pytest

import oracle
from blas_helpers import U32, bound_ratio
from clgpu_amd import datagen
from clgpu_amd import iclblas as ib
from l3_helpers import RANK2K, RANKK, call_library, oracle_result, random_case, shapes

pytestmark = pytest.mark.gpu
REAL = [n for n in ib.implementation_names() if n.startswith("sgemm_f32_split3")]
CPLX = [n for n in ib.implementation_names() if n.startswith("cgemm_f32_split3")]


@pytest.fixture
def h(handle):
    handle.set_math_mode(ib.MATH_FP32)
    yield handle
    handle.set_implementation(None)


def _dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x.T)).cuda()


# one slab, a partial slab, the ring's start-up lengths (2, 3, 4 slabs), depths that are
# split over workgroups (into equal and unequal parts, by 4 and by more than 8); one row
# past a tile and one short of it
SHAPES = [(1, 1, 1), (127, 129, 31), (129, 127, 33), (256, 128, 64), (255, 257, 96), (300, 70, 128), (128, 256, 417),
          (257, 129, 2048), (130, 127, 5000)]


@pytest.mark.parametrize("impl", REAL)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_real_edges(h, impl, ta, tb, shape):
    m, n, k = shape
    ra, ca = (m, k) if ta == 0 else (k, m)
    rb, cb = (k, n) if tb == 0 else (n, k)
    A = datagen.matrix(ra, ca, ra + 3, "A", seed=41)
    B = datagen.matrix(rb, cb, rb + 1, "B", seed=41)
    C = datagen.matrix(m, n, m + 2, "C", seed=41)
    A[ra:], B[rb:] = np.nan, np.nan  # padding rows are never read
    C0 = C.copy(order="F")
    C64, ab = oracle.dgemm(ta, tb, m, n, k, -1.5, A, B, 0.5, C)
    h.set_implementation(impl)
    ib.check(ib.iclblasSgemm(h.value, ta, tb, m, n, k, -1.5, A, ra + 3, B, rb + 1, 0.5, C, m + 2))
    assert h.last_implementation() == impl
    extra = 2 * U32 * (0.5 * np.abs(C0[:m].astype(np.float64)) + 1.5 * ab)
    assert bound_ratio(np.abs(C[:m].astype(np.float64) - C64), k, 1.5 * ab, extra) <= 4.0
    assert np.array_equal(C[m:], C0[m:])


@pytest.mark.parametrize("impl", CPLX)
@pytest.mark.parametrize("ta", [0, 1, 2])
@pytest.mark.parametrize("tb", [0, 1, 2])
@pytest.mark.parametrize("shape", [(1, 1, 1), (63, 129, 15), (65, 127, 17), (129, 257, 48), (128, 70, 65), (65, 129, 1500)],
                         ids=lambda s: "x".join(map(str, s)))
def test_complex_edges(h, impl, ta, tb, shape):
    m, n, k = shape
    ra, ca = (m, k) if ta == 0 else (k, m)
    rb, cb = (k, n) if tb == 0 else (n, k)
    A = datagen.complex_matrix(ra, ca, ra + 1, "A", seed=42)
    B = datagen.complex_matrix(rb, cb, rb + 2, "B", seed=42)
    C = datagen.complex_matrix(m, n, m + 1, "C", seed=42)
    alpha, beta = 1 + 0.5j, 0.25 - 0.5j
    C0 = C.copy(order="F")
    C64, ab = oracle.zgemm(ta, tb, m, n, k, alpha, A, B, beta, C)
    h.set_implementation(impl)
    ib.check(ib.iclblasCgemm(h.value, ta, tb, m, n, k, alpha, A, ra + 1, B, rb + 2, beta, C, m + 1))
    assert h.last_implementation() == impl
    extra = 4 * U32 * (abs(beta) * np.abs(C0[:m]).astype(np.float64) + abs(alpha) * ab)
    assert bound_ratio(np.abs(C[:m].astype(np.complex128) - C64), k, abs(alpha) * ab, extra) <= 4.0
    assert np.array_equal(C[m:], C0[m:])


LEVEL3 = [("Ssyrk", dict(uplo=0, trans=1), (None, 300, 70)), ("Ssyrk", dict(uplo=1, trans=1), (None, 600, 1500)),
          ("Cherk", dict(uplo=0, trans=0), (None, 140, 700)), ("Strmm", dict(side=0, uplo=1, trans=0, diag=0), (700, 130, None)),
          ("Ssyrk", dict(uplo=1, trans=0), (None, 256, 33)),
          ("Ssyrk", dict(uplo=0, trans=0), (None, 513, 33)), ("Csyrk", dict(uplo=0, trans=0), (None, 641, 16)),
           ("Cherk", dict(uplo=1, trans=0), (None, 513, 16)),
          ("Ssyr2k", dict(uplo=1, trans=1), (None, 259, 64)), ("Cherk", dict(uplo=0, trans=2), (None, 140, 65)),
          ("Csyrk", dict(uplo=0, trans=2), (None, 130, 40)),
          ("Cher2k", dict(uplo=1, trans=0), (None, 128, 40)), ("Ssymm", dict(side=1, uplo=0), (130, 290, None)),
          ("Chemm", dict(side=0, uplo=1), (150, 70, None))] + [
    (r, dict(side=s, uplo=u, trans=t, diag=d), (270, 140, None) if s == 0 else (140, 270, None))
    for r in ("Strmm", "Ctrmm") for s in (0, 1) for u in (0, 1) for t, d in ((0, 0), (2, 1))]


@pytest.mark.parametrize("tile", [0, 1])
@pytest.mark.parametrize("routine,v,shape", LEVEL3, ids=lambda x: str(x).replace(" ", ""))
def test_level3_options(h, routine, v, shape, tile):
    m, n, k = shape
    c = random_case(routine, np.random.default_rng(n), m=m, n=n, k=k, **v)
    impl = (CPLX if routine[0] == "C" else REAL)[tile]
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


def _native(fn):
    """The same call on a handle whose scratch cap keeps it on FP32 MFMA."""
    import torch
    with ib.Handle(memory_mode=ib.MEMORY_DEVICE, stream=torch.cuda.current_stream().cuda_stream) as hn:
        hn.set_scratch_limit(1 << 40)
        fn(hn)
        torch.cuda.synchronize()
        assert "split3" not in hn.last_implementation()


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4e38, 2.0 ** 50, 2.0 ** -111, 1e-45])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("where", ["A", "B"])
def test_guard_gives_the_fp32_result(dev_handle, value, cplx, where):
    """One element outside the split's range: bit for bit the FP32 MFMA result, on
    several calls in a row (the guard word is not cleared between them), and the
    split kernel again once the operand is back in range."""
    import torch
    h = dev_handle
    h.set_math_mode(ib.MATH_FP32)
    h.set_implementation(None)
    m = n = k = 2048
    make = datagen.complex_matrix if cplx else datagen.matrix
    call = ib.iclblasCgemm if cplx else ib.iclblasSgemm
    tA, tB = _dev(make(m, k, name="A", seed=43)), _dev(make(k, n, name="B", seed=43))
    C0 = _dev(make(m, n, name="C", seed=43))
    t = tA if where == "A" else tB
    kept = t[700, 901].clone()

    def run(hh, C):
        ib.check(call(hh.value, 0, 0, m, n, k, 1.0, tA, m, tB, k, 0.5, C, m))

    t[700, 901] = complex(0.5, value) if cplx else value
    for _ in range(2):
        C, D = C0.clone(), C0.clone()
        run(h, C)
        assert "split3" in h.last_implementation()
        _native(lambda hn: run(hn, D))
        bits = lambda t: (torch.view_as_real(t) if cplx else t).view(torch.int32)  # noqa: E731
        assert torch.equal(bits(C), bits(D))
    t[700, 901] = kept
    C, D = C0.clone(), C0.clone()
    run(h, C)
    torch.cuda.synchronize()
    assert bool(torch.isfinite(torch.view_as_real(C) if cplx else C).all())
    _native(lambda hn: run(hn, D))
    assert not torch.equal(C, D)  # (its accuracy is checked above)


def test_capture_stays_on_fp32_mfma():
    """A captured call takes no optional workspace: the graph holds only the FP32
    MFMA kernel, and replays match after other, larger products have run."""
    import torch
    n = 2048
    tA, tB = _dev(datagen.matrix(n, n, name="A", seed=44)), _dev(datagen.matrix(n, n, name="B", seed=44))
    C, D, E = (torch.empty((n, n), device="cuda") for _ in range(3))
    side = torch.cuda.Stream()
    with ib.Handle(memory_mode=ib.MEMORY_DEVICE, stream=side.cuda_stream) as h:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            ib.check(ib.iclblasSgemm(h.value, 0, 0, n, n, n, 1.0, tA, n, tB, n, 0.0, C, n))
        assert "split3" not in h.last_implementation()
        _native(lambda hn: ib.check(ib.iclblasSgemm(hn.value, 0, 0, n, n, n, 1.0, tA, n, tB, n, 0.0, D, n)))
        for _ in range(3):
            C.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(C, D)
            ib.check(ib.iclblasSgemm(h.value, 0, 1, n, n, n, 1.0, tA, n, tB, n, 0.0, E, n))
            h.synchronize()


@pytest.mark.parametrize("impl", REAL)
def test_sums_of_squares_lose_nothing(h, impl):
    """A A^T's diagonal sums products whose small parts are squares too: cut off instead of rounded they
    would leave every sum short. The mean error over 4096 sums of 32 slabs: at most 2^-23 from the terms
    left out, and five standard deviations of 32 roundings to nearest averaged over 4096 sums."""
    import torch
    n, k = 4096, 1024
    A = torch.empty((k, n), device="cuda").uniform_(-1, 1, generator=torch.Generator("cuda").manual_seed(5))
    C = torch.empty((n, n), device="cuda")
    E = (A.double() ** 2).sum(0)
    h.set_memory_mode(ib.MEMORY_DEVICE)
    h.set_implementation(impl)
    torch.cuda.synchronize()
    try:
        ib.check(ib.iclblasSgemm(h.value, 0, 1, n, n, k, 1.0, A, n, A, n, 0.0, C, n))
        h.synchronize()
    finally:
        h.set_memory_mode(ib.MEMORY_HOST)
    off = ((C.diag().double() - E) / E).mean().abs().item()
    assert off <= 2.0 ** -23 + 5 * U32 * (k / 32) ** 0.5 / n ** 0.5


def _split_handle(cap):
    import torch
    h = ib.Handle(memory_mode=ib.MEMORY_DEVICE, math_mode=ib.MATH_SPLIT_BF16X3,
                  stream=torch.cuda.current_stream().cuda_stream)
    h.set_scratch_limit(cap)
    return h


@pytest.mark.parametrize("cplx,n,cap,impl", [
    (False, 1024, 8 << 20, "sgemm_bf16x3d"),  # just the packed operands, no partial sums
    (True, 2048, 80 << 20, "cgemm_bf16x3_"),  # 64 MiB packed once, 96 MiB with op(A) packed as rows of two
    (True, 2048, 96 << 20, "cgemm_bf16x3d"),
    (True, 2048, 60 << 20, None)])
def test_split_bf16_under_a_cap(cplx, n, cap, impl):
    """A capped handle's split-BF16 products: what the packed operands fit runs, what they do not is refused."""
    rnd = np.random.default_rng(8)
    A, B = (rnd.standard_normal((n, n)).astype(np.float32) for _ in range(2))
    if cplx:
        A, B = (X + 1j * rnd.standard_normal((n, n)).astype(np.float32) for X in (A, B))
    tA, tB = _dev(A), _dev(B)
    import torch
    C = torch.zeros_like(tA)
    with _split_handle(cap) as h:
        f = ib.iclblasCgemm if cplx else ib.iclblasSgemm
        st = f(h.value, 0, 0, n, n, n, 1.0, tA.data_ptr(), n, tB.data_ptr(), n, 0.0, C.data_ptr(), n)
        h.synchronize()
        if impl is None:
            assert st == ib.STATUS_ALLOC_FAILED and not C.any()
            return
        ib.check(st)
        assert h.last_implementation().startswith(impl)
        assert h.scratch_usage()[0] <= cap
    W = np.complex128 if cplx else np.float64
    E = A.astype(W) @ B.astype(W)
    ab = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)
    c = 2 if cplx else 1
    assert bound_ratio(np.abs(C.cpu().numpy().T.astype(W) - E), c * n, c * ab) <= 4.0
