"""Memory that only makes a call faster (the packed operands of the split kernels) against the
calls that need memory: a handle's cap, a captured stream, the static scratch."""
import numpy as np
import pytest

from clgpu_amd import datagen
from clgpu_amd import iclblas as ib

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
