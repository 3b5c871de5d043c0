"""Memory that only makes a call faster (the packed operands of the split kernels) against the
calls that need memory: a handle's cap, a captured stream, the static scratch."""
import numpy as np
import pytest

from blas_helpers import U32
from clgpu_amd import datagen
from clgpu_amd import iclblas as ib
from l3_helpers import RANK2K, RANKK, call_library, oracle_result, random_case, shapes

pytestmark = pytest.mark.gpu


def _handle(mode=ib.MATH_FP32, stream=None):
    import torch
    stream = torch.cuda.current_stream() if stream is None else stream
    return ib.Handle(memory_mode=ib.MEMORY_DEVICE, math_mode=mode, stream=stream.cuda_stream)


def _dev(x):
    import torch
    return torch.from_numpy(np.ascontiguousarray(x.T)).cuda()


def _sgemm(h, n, tA, tB, tC, m=None, k=None):
    m, k = m or n, k or n
    ib.check(ib.iclblasSgemm(h.value, 0, 0, m, n, k, 1.0, tA, m, tB, k, 0.0, tC, m))


def test_optional_memory_gives_way_to_a_cap():
    """What an uncapped FP32 product took does not count against buffers that a call needs under a cap
    set later; a call that the cap refuses all the same frees nothing."""
    import torch
    n, nr = 1024, 256
    tA, tB, tC = (torch.rand((2048, 2048), device="cuda") for _ in range(3))
    T = datagen.triangular(n, lower=True, seed=5)
    tT, tX = _dev(T), _dev(datagen.matrix(n, nr, name="B", seed=5))
    tY = tX.clone()
    with _handle() as h:
        _sgemm(h, 2048, tA, tB, tC)
        h.synchronize()
        assert "split3" in h.last_implementation()
        held = h.scratch_usage()[0]
        assert held > 32 << 20
        h.set_scratch_limit(64 << 10)
        st = ib.iclblasStrsm(h.value, 0, 1, 0, 0, n, nr, 1.0, tT, n, tX, n)
        assert st == ib.STATUS_ALLOC_FAILED and h.scratch_usage()[0] == held
        h.set_scratch_limit(16 << 20)
        ib.check(ib.iclblasStrsm(h.value, 0, 1, 0, 0, n, nr, 1.0, tT, n, tX, n))
        h.synchronize()
        assert h.scratch_usage()[0] <= 16 << 20
    with _handle() as h:
        h.set_scratch_limit(16 << 20)
        ib.check(ib.iclblasStrsm(h.value, 0, 1, 0, 0, n, nr, 1.0, tT, n, tY, n))
        h.synchronize()
    assert torch.equal(tX, tY)


@pytest.mark.parametrize("routine,v,shape,packed_once", [
    # n = 640, k = 700: 2 * 640 * 704 * 8 bytes = 6.9 MiB packed once, 10.3 with op(A) as rows of two
    ("Cherk", dict(uplo=1, trans=0), (None, 640, 700), 2 * 640 * 704 * 8),
    ("Csyrk", dict(uplo=0, trans=2), (None, 640, 700), 2 * 640 * 704 * 8),
    ("Cher2k", dict(uplo=0, trans=2), (None, 640, 700), 2 * 640 * 704 * 8),
    ("Ctrmm", dict(side=0, uplo=1, trans=0, diag=0), (640, 512, None), (640 + 512) * 640 * 8 + 640 * 640 * 8),
    ("Ctrmm", dict(side=1, uplo=0, trans=2, diag=1), (512, 640, None), (640 + 512) * 640 * 8 + 640 * 640 * 8),
])
def test_complex_level3_under_a_cap(routine, v, shape, packed_once):
    """Split-BF16 updates whose operands fit the cap packed once, but not with op(A) packed as rows of
    two parts, run; a cap below that refuses them."""
    import torch
    m, n, k = shape
    c = random_case(routine, np.random.default_rng(11), m=m, n=n, k=k, **v)
    (rc, cc) = shapes(c)[2]
    tA, tB, tC = (None if c.get(x) is None else _dev(c[x]) for x in "ABC")
    ptr = [t if t is None else t.data_ptr() for t in (tA, tB)]
    for cap, status in ((packed_once - (1 << 20), ib.STATUS_ALLOC_FAILED), (packed_once + (1 << 20), ib.STATUS_SUCCESS)):
        with _handle(ib.MATH_SPLIT_BF16X3) as h:
            h.set_scratch_limit(cap)
            assert call_library(h.value, c, ptr[0], ptr[1], tC.data_ptr()) == status
            h.synchronize()
            assert h.scratch_usage()[0] <= cap
        if status != ib.STATUS_SUCCESS:
            assert np.array_equal(tC.cpu().numpy().T, c["C"], equal_nan=True)
    C = tC.cpu().numpy().T
    exp, mag, kk = oracle_result(c, c["A"], c.get("B"), c["C"])
    written = np.ones((rc, cc), bool)
    if routine in RANKK or routine in RANK2K:
        written = np.tril(written) if v["uplo"] == 1 else np.triu(written)
    C0 = np.abs(np.nan_to_num(c["C"][:rc, :cc].astype(np.complex128)))
    bound = 4.0 * (2 * kk + 2) * U32 * (abs(c["alpha"]) * mag + abs(c.get("beta", 0.0)) * C0)
    err = np.abs(C[:rc, :cc].astype(np.complex128) - exp[:rc, :cc])
    assert np.all((err <= bound)[written])
    assert np.array_equal(C[:rc, :cc][~written], c["C"][:rc, :cc][~written])
    torch.cuda.synchronize()


def _split_product(h, cplx, m, n, k, call=None):
    """A product in the split-BF16 mode on device memory: (status, check of the result)."""
    import torch
    gen = torch.Generator("cuda").manual_seed(13)
    dt = torch.complex64 if cplx else torch.float32
    A, B = (torch.rand(s, device="cuda", generator=gen, dtype=dt) - 0.5 for s in ((k, m), (n, k)))
    C = torch.full((n, m), float("nan"), device="cuda", dtype=dt)
    torch.cuda.synchronize()
    call = call or (ib.iclblasCgemm if cplx else ib.iclblasSgemm)

    def run():
        return call(h.value, 0, 0, m, n, k, 1.0, A.data_ptr(), m, B.data_ptr(), k, 0.0, C.data_ptr(), m)

    def check():
        wide = torch.complex128 if cplx else torch.float64
        err = (C.to(wide) - B.to(wide) @ A.to(wide)).abs()
        kk = 2 * k if cplx else k
        assert bool((err <= 4 * kk * U32 * (2 if cplx else 1) * (B.abs().double() @ A.abs().double())).all())
    return run, check, C


# (complex, m, n, k, bytes): what a split-BF16 product requires is part of the library's behaviour under
# a cap. Operands packed once, rows in tiles of 128 or 256, or nothing: several of the latter run on the
# packed kernels where memory is free.
REQUIRED = [(False, 1024, 1024, 1024, 8388608), (False, 700, 900, 300, 2293760), (False, 1280, 2944, 1280, 21626880),
            (False, 130, 4000, 3000, 52363264), (True, 640, 700, 512, 0), (True, 1030, 1111, 300, 0),
            (True, 1664, 512, 641, 0), (True, 2304, 2048, 335, 0), (True, 1500, 1400, 1300, 30900224),
            (True, 129, 3000, 2000, 0)]


@pytest.mark.parametrize("cplx,m,n,k,required", REQUIRED)
def test_required_workspace_under_a_cap(cplx, m, n, k, required):
    import torch
    if required:
        with _handle(ib.MATH_SPLIT_BF16X3) as h:
            run, _, C = _split_product(h, cplx, m, n, k)
            h.set_scratch_limit(required - 1)
            assert run() == ib.STATUS_ALLOC_FAILED
            h.synchronize()
            assert bool(torch.isnan(C).all())
    for cap in (max(required, 256), 3 * required + (64 << 10)):
        with _handle(ib.MATH_SPLIT_BF16X3) as h:
            run, check, _ = _split_product(h, cplx, m, n, k)
            h.set_scratch_limit(cap)
            ib.check(run())
            h.synchronize()
            check()
            assert "bf16x3" in h.last_implementation() and h.scratch_usage()[0] <= cap


@pytest.mark.parametrize("m,n,k", [(2304, 2048, 335), (1664, 512, 641)])
def test_captured_product_that_requires_nothing(m, n, k):
    """Captured without a call before it on that handle: it may not allocate."""
    import torch
    side = torch.cuda.Stream()
    with _handle(ib.MATH_SPLIT_BF16X3, side) as h:
        run, check, C = _split_product(h, True, m, n, k)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            ib.check(run())
        assert h.scratch_usage()[0] == 0
        for _ in range(3):
            C.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            check()


def test_no_alloc_takes_the_variant_that_fits():
    """4608 x 2944 x 2208: 63.6 MiB of packed operands in rows of 128, 64.7 in rows of 256."""
    m, n, k = 4608, 2944, 2208
    with _handle(ib.MATH_SPLIT_BF16X3) as h:
        run, check, _ = _split_product(h, False, m, n, k, ib.iclblasSgemmNoAlloc)
        ib.check(run())
        h.synchronize()
        check()
        assert h.last_implementation().startswith("sgemm_bf16x3d") and h.scratch_usage()[0] == 0


def test_a_graph_keeps_its_workspace():
    """A captured product, then one that requires no more but would like partial sums: its larger workspace
    is not the one that the graph holds."""
    import torch
    side = torch.cuda.Stream()
    with _handle(ib.MATH_SPLIT_BF16X3, side) as h:
        run, check, C = _split_product(h, False, 4096, 4096, 1024)  # packed: 32 MiB
        ib.check(run())
        h.synchronize()
        held = h.scratch_usage()[0]
        assert held == 32 << 20
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            ib.check(run())
        with _handle(ib.MATH_SPLIT_BF16X3) as other:
            ib.check(_split_product(other, False, 1024, 1024, 4096)[0]())
            other.synchronize()
            more = other.scratch_usage()[0]
        assert more > held  # packed: 32 MiB, and partial sums
        run2, check2, _ = _split_product(h, False, 1024, 1024, 4096)
        ib.check(run2())
        h.synchronize()
        assert h.scratch_usage()[0] == held + more
        check2()
        fill = torch.full((64 << 20,), float("nan"), device="cuda")
        for _ in range(3):
            C.fill_(float("nan"))
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            check()
            ib.check(run2())
            h.synchronize()
            check2()
        del fill


def test_optional_memory_leaves_a_capture_alone():
    """FP32 products on a stream of their own while another stream is captured: they take their optional
    workspace, the second a larger one, and the capture stays valid."""
    import torch
    n = 2048
    tA, tB, tC, tD = (torch.rand((2 * n, n), device="cuda") for _ in range(4))
    x = torch.zeros(1024, device="cuda")
    captured, other = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with _handle(stream=other) as h:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=captured):
            x += 1
            _sgemm(h, n, tA, tB, tC)
            assert "split3" in h.last_implementation()
            held = h.scratch_usage()[0]
            _sgemm(h, n, tA, tB, tD, m=2 * n)
            assert h.scratch_usage()[0] > held > 0
            x += 1
        h.synchronize()
        for i in range(3):
            graph.replay()
            torch.cuda.synchronize()
            assert bool((x == 2 * (i + 1)).all())
    E = (tB[:n].double() @ tA[:n].double())
    assert bool(((tC[:n] - E).abs() <= 4 * n * U32 * E).all())


def test_no_alloc_in_the_fp32_mode():
    """Where iclblasSgemm takes the packed kernels: FP32 MFMA, no memory, a result within the same bound."""
    for call, name in ((ib.iclblasSgemm, "split3"), (ib.iclblasSgemmNoAlloc, "sgemm_f32_")):
        with _handle() as h:
            run, check, _ = _split_product(h, False, 2048, 2048, 2048, call)
            ib.check(run())
            h.synchronize()
            check()
            assert name in h.last_implementation()
            assert ("split3" in h.last_implementation()) == (h.scratch_usage()[0] > 0) == (call is ib.iclblasSgemm)
