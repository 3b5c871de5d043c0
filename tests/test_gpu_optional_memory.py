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
