"""The packed split kernels beyond 32-bit sizes: operands of more rows than a 32-bit extent
of one slab reaches, and depths of more slabs than a grid's second dimension holds."""
import pytest

from blas_helpers import U32
from clgpu_amd import iclblas as ib

pytestmark = pytest.mark.gpu


def _call(impl, ta, tb, m, n, k, A, lda, B, ldb, C, ldc):
    """One SGEMM with `impl` on a handle of its own."""
    import torch
    mode = ib.MATH_SPLIT_BF16X3 if "bf16x3" in impl else ib.MATH_FP32
    with ib.Handle(memory_mode=ib.MEMORY_DEVICE, math_mode=mode, stream=torch.cuda.current_stream().cuda_stream) as h:
        h.set_implementation(impl)
        ib.check(ib.iclblasSgemm(h.value, ta, tb, m, n, k, 1.0, A, lda, B, ldb, 0.0, C, ldc))
        h.synchronize()
        assert h.last_implementation() == impl


@pytest.mark.parametrize("impl", [n for n in ib.implementation_names()
                                  if n.startswith(("sgemm_f32_split3", "sgemm_bf16x3d"))])
def test_rows_past_the_32_bit_extent_of_a_slab(impl):
    """2^25 + 130 rows: a slab of two planes is 4 GiB and one tile, of three planes 6 GiB. Sampled rows
    against float64, in the first tile, on both sides of every 2^24 rows and in the last, ragged one."""
    import torch
    m, n, k = (1 << 25) + 130, 3, 256
    gen = torch.Generator("cuda").manual_seed(6)
    A = torch.empty((k, m), device="cuda")  # op(A) = A, column major
    for i in range(0, k, 32):
        A[i:i + 32].uniform_(-1, 1, generator=gen)
    B = torch.empty((n, k), device="cuda").uniform_(-1, 1, generator=gen)
    C = torch.full((n, m), float("nan"), device="cuda")
    torch.cuda.synchronize()
    _call(impl, 0, 0, m, n, k, A, m, B, k, C, m)
    rows = [r for c in (0, 1 << 22, 1 << 24, 3 << 23, m - 130, m) for r in range(c - 260, c + 260) if 0 <= r < m]
    rows = torch.tensor(rows + list(range(0, m, 65521)), device="cuda")
    X, Y = A[:, rows].double(), B.double()
    err, mag = (C[:, rows].double() - Y @ X).abs(), Y.abs() @ X.abs()
    assert bool((err <= 4 * k * U32 * mag).all())
    assert bool(torch.isfinite(C).all())
    del A, B, C, X
    torch.cuda.empty_cache()


@pytest.mark.parametrize("impl", ["sgemm_f32_split3_128x128", "sgemm_bf16x3d_mfma_128x128"])
@pytest.mark.parametrize("ta,tb", [(0, 1), (1, 0)])
def test_depth_past_the_grid_limit(impl, ta, tb):
    """k = 2^22 + 100: 65538 pairs of slabs."""
    import torch
    m, n, k = 60, 70, (1 << 22) + 100
    gen = torch.Generator("cuda").manual_seed(7)
    A, B = (torch.empty((r, c), device="cuda").uniform_(-1, 1, generator=gen)
            for r, c in (((k, m) if ta == 0 else (m, k)), ((n, k) if tb == 0 else (k, n))))
    C = torch.full((n, m), float("nan"), device="cuda")
    torch.cuda.synchronize()
    _call(impl, ta, tb, m, n, k, A, A.shape[1], B, B.shape[1], C, m)
    X, Y = (A.T if ta == 0 else A).double(), (B.T if tb == 0 else B).double()
    err, mag = (C.T.double() - X @ Y).abs(), X.abs() @ Y.abs()
    assert bool((err <= 4 * k * U32 * mag).all())
    # the bound above grows with k: the last slabs, alone in a block of rows of zeros
    A[(slice(0, 1 << 22), 0) if ta == 0 else (0, slice(0, 1 << 22))] = 0
    _call(impl, ta, tb, m, n, k, A, A.shape[1], B, B.shape[1], C, m)
    X = (A.T if ta == 0 else A).double()
    err, mag = (C.T.double() - X @ Y).abs()[0], (X.abs() @ Y.abs())[0]
    assert bool((err <= 4 * 256 * U32 * mag).all())
