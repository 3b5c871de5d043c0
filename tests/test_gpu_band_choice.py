"""Triangle updates as two launches (off the diagonal blocks, on them): only where both are tiled kernels,
whose model chose the pair. Few shallow tiles run the triangle whole, whatever kernel that is."""
import pytest

from blas_helpers import U32
from clgpu_amd import iclblas as ib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("trans", [0, 1])
@pytest.mark.parametrize("uplo", [0, 1])
@pytest.mark.parametrize("n,k", [(825, 104), (600, 60), (1000, 40), (700, 90), (3008, 128)])
def test_pair_is_tiled(n, k, uplo, trans):
    import torch
    A = torch.rand((k, n) if trans == 0 else (n, k), device="cuda") - 0.5
    C0 = torch.rand((n, n), device="cuda")
    C = C0.clone()
    with ib.Handle(memory_mode=ib.MEMORY_DEVICE, stream=torch.cuda.current_stream().cuda_stream) as h:
        h.set_kernel_timing(True)
        ib.check(ib.iclblasSsyrk(h.value, uplo, trans, n, k, 1.0, A, A.shape[1], 0.5, C, n))
        launches = h.kernel_timing()[1]
        assert launches == 1 or (launches == 2 and "wave" not in h.last_implementation())
    X = A.double() if trans == 0 else A.double().T
    E, mag = X.T @ X + 0.5 * C0.double(), X.abs().T @ X.abs() + 0.5 * C0.double()
    written = torch.ones_like(C, dtype=torch.bool)
    written = written.tril() if uplo == 0 else written.triu()  # torch's rows are columns
    assert bool(((C - E).abs() <= 4 * (k + 2) * U32 * mag)[written].all())
    assert torch.equal(C[~written], C0[~written])
