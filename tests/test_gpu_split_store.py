"""The checked stores of the packed split kernels: a triangle mask (zeros outside it) at the
edges of the tiles."""
import numpy as np
import pytest

from blas_helpers import U32
from clgpu_amd import datagen
from clgpu_amd import iclblas as ib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("impl", [n for n in ib.implementation_names() if n.startswith("sgemm_f32_split3")])
@pytest.mark.parametrize("order", [129, 383])
@pytest.mark.parametrize("uplo", [0, 1])
@pytest.mark.parametrize("diag", [0, 1])
@pytest.mark.parametrize("trans", [0, 1])
def test_masked_product(handle, impl, order, uplo, diag, trans):
    """The gradient of a triangular solve with the identity: dA = -dX X^T (or its transpose) in the
    stored triangle, without the diagonal of a unit one, and zeros elsewhere."""
    n, ld = 70, order + 3
    A = np.asfortranarray(np.eye(order, dtype=np.float32))
    X, dX = (datagen.matrix(order, n, name=s, seed=45) for s in "AB")
    dA = np.full((ld, order), 7.0, np.float32, order="F")
    handle.set_math_mode(ib.MATH_FP32)
    handle.set_implementation(impl)
    try:
        ib.check(ib.iclblasStrsmBackward(handle.value, 0, uplo, trans, diag, order, n, 1.0, A, order, X, order, dX,
                                         order, dA, ld, None, order))
    finally:
        handle.set_implementation(None)
    L, R = (dX, X) if trans == 0 else (X, dX)
    E = -L.astype(np.float64) @ R.astype(np.float64).T
    mag = np.abs(L).astype(np.float64) @ np.abs(R).astype(np.float64).T
    keep = np.tril(np.ones((order, order), bool)) if uplo == 1 else np.triu(np.ones((order, order), bool))
    if diag == 1:
        np.fill_diagonal(keep, False)
    got = dA[:order]
    assert np.all((np.abs(got - E) <= 4 * n * U32 * mag)[keep])
    assert np.all(got[~keep] == 0.0) and np.all(dA[order:] == 7.0)
