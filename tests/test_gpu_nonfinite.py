"""Infinities beside zeros: a chain with an all-zero factor has norm 0, and a
dense product of 64K entries or more leaves the zeros of a sparse operand out
whatever its size."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

import faust_amd
from faust_amd import _lib, fact, factparams

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [24, 300])  # the power iteration's forms: LDS, past it
@pytest.mark.parametrize("r2l", [False, True])
def test_zero_factor_beside_infinities(gpu, n, r2l):
    # the first step size is taken from the two other factors, one of them all zeros and not counted before
    rng = np.random.default_rng(n)
    inf = rng.standard_normal((n, n))
    inf[rng.integers(0, n, 5), rng.integers(0, n, 5)] = np.inf
    other = [np.zeros((n, n)), np.asfortranarray(inf)]
    facs = other + [np.eye(n)] if r2l else [np.eye(n)] + other
    cons = [factparams.ConstraintInt("sp", n, n, 4 * n)] * 3
    p = factparams.ParamsPalm4MSA(cons, factparams.StoppingCriterion(num_its=2), factor_format="dense",
                                  packing_RL=False, is_update_way_R2L=r2l)
    # the C entry points, since faust_amd.Faust has its factors counted when it is made
    init, out, keep = C.c_void_p(), C.c_void_p(), []
    _lib.check(gpu.fh_faust_create(C.byref(init)))
    handles = [faust_amd.Factor(f) for f in facs]
    for h in handles:
        _lib.check(gpu.fh_faust_push_back(init, h.h))
    A = np.asfortranarray(rng.standard_normal((n, n)))
    cc = (_lib.fh_constraint * 3)(*[c._c(keep) for c in p.constraints])
    sc, pc = p.stop_crit._c(), p._c(False)
    with pytest.raises(_lib.FaustHipError, match="2-norm is zero"):
        _lib.check(gpu.fh_palm4msa(A.ctypes.data_as(C.c_void_p), n, n, cc, 3, C.byref(sc), C.byref(pc), 1.0, init,
                                   C.byref(out)))
    _lib.check(gpu.fh_faust_free(init))


@pytest.mark.parametrize("n", [256, 300, 723, 724, 900])  # 64K, and both sides of 512K entries
@pytest.mark.parametrize("sides", ["left", "right", "three"])
def test_zeros_against_infinities_in_products(gpu, n, sides):
    rng = np.random.default_rng(n)
    S = rng.standard_normal((n, n)) * (rng.random((n, n)) < 0.03)
    S[:, 3] = S[3, :] = 0.0
    D = rng.standard_normal((n, n))
    D[3, 5] = np.inf  # meets zeros only, on either side
    D[5, 3] = -np.inf
    E = rng.standard_normal((n, n))
    facs = {"left": [S, D], "right": [D, S], "three": [E, S, D]}[sides]
    got = faust_amd.Faust([np.asfortranarray(f) for f in facs]).toarray()
    Sc = sp.csr_matrix(S)
    with np.errstate(invalid="ignore"):
        want = {"left": lambda: Sc @ D, "right": lambda: (Sc.T @ D.T).T, "three": lambda: E @ np.asarray(Sc @ D)}[sides]()
    want = np.asarray(want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    fin = np.isfinite(want)
    assert fin.sum() > n and np.array_equal(got[~fin], want[~fin], equal_nan=True)
    # sums of at most 2 n terms in another order
    bound = np.eye(n)
    for f in facs:
        bound = bound @ np.where(np.isfinite(f), np.abs(f), 0.0)
    assert np.all(np.abs(got[fin] - want[fin]) <= 4 * n * 2.0 ** -53 * bound[fin])
