"""k_gemm_f64's tile edges and K remainders bit for bit against the oracle: one
shape per tile choice and side of it, with denormals, infinities, exact zeros
and values far apart in the operands."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
from faust_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opA,opB", [("N", "N"), ("T", "N"), ("N", "T"), ("T", "T")])
@pytest.mark.parametrize("mnk", [(31, 33, 1), (32, 65, 31), (17, 1, 1025), (800, 832, 33), (801, 801, 4),
                                 (1793, 1760, 5)])
def test_gemm_tiles_bitexact(gpu, opA, opB, mnk):
    m, n, k = mnk
    rng = np.random.default_rng(m + k)

    def draw(r, c):
        a = rng.standard_normal((r, c)) * np.exp2(rng.integers(-60, 60, (r, c)))
        a[rng.random((r, c)) < 0.05] = 0.0
        a[rng.integers(0, r, 2), rng.integers(0, c, 2)] = [5e-324, -1e-310]
        return np.asfortranarray(a)

    A = draw(*((m, k) if opA == "N" else (k, m)))
    B = draw(*((k, n) if opB == "N" else (n, k)))
    # the infinity meets nonzero terms only: the oracle skips exact zeros, so 0 x inf has no canonical value
    A[0, 0] = np.inf
    line = B[0, :] if opB == "N" else B[:, 0]
    line[line == 0.0] = 1.0
    C0 = np.asfortranarray(rng.standard_normal((m, n)))
    dA, dB = (torch.from_numpy(np.ascontiguousarray(x.T)).cuda() for x in (A, B))
    dC = torch.from_numpy(np.ascontiguousarray(C0.T)).cuda()
    a, b = C.c_double(-0.7), C.c_double(1.0)
    _lib.check(gpu.fh_gemm(_lib.FH_F64, opA.encode(), opB.encode(), m, n, k, C.byref(a), C.c_void_p(dA.data_ptr()),
                           A.shape[0], C.c_void_p(dB.data_ptr()), B.shape[0], C.byref(b), C.c_void_p(dC.data_ptr()),
                           m, None))
    torch.cuda.synchronize()
    with np.errstate(invalid="ignore"):
        assert np.array_equal(dC.cpu().numpy().T, oracle.gemm(A, B, opA, opB, -0.7, 1.0, C0), equal_nan=True)
