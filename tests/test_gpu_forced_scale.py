"""Level-3 updates with alpha = 0, a product of depth 0, with every GEMM implementation chosen by
name: beta C in the written triangle, A never read."""
import numpy as np
import pytest

from clgpu_amd import iclblas as ib
from l3_helpers import call_library, closed_form, random_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [ib.MATH_FP32, ib.MATH_SPLIT_BF16X3])
@pytest.mark.parametrize("impl", [n for n in ib.implementation_names() if "gemm" in n])
def test_alpha_zero(handle, impl, mode):
    routines = (("Cherk", dict(uplo=1, trans=0)), ("Csymm", dict(side=0, uplo=0))) if impl[0] == "c" else (
        ("Ssyrk", dict(uplo=0, trans=1)), ("Ssymm", dict(side=1, uplo=1)))
    handle.set_math_mode(mode)
    handle.set_implementation(impl)
    try:
        for routine, v in routines:
            m, n, k = (None, 131, 300) if "k" in routine else (131, 67, None)
            c = random_case(routine, np.random.default_rng(3), m=m, n=n, k=k, alpha=0.0, beta=0.5, **v)
            A, B, C = (None if c.get(x) is None else c[x].copy(order="F") for x in "ABC")
            ib.check(call_library(handle.value, c, A, B, C), routine)
            A0, B0 = (None if c.get(x) is None else np.zeros_like(c[x]) for x in "AB")
            assert np.array_equal(C, closed_form(c, A0, B0, c["C"]).astype(C.dtype))
    finally:
        handle.set_implementation(None)
        handle.set_math_mode(ib.MATH_FP32)
