"""The kernels between PALM4MSA's products, at the sizes where they can go
wrong, bit for bit against the oracle: the sp selection (candidate list full,
ties past it, every digit needed), line selections that keep whole lines, the
tiles of the dense -> CSR conversion, the diagonal of A^T S, and the zero
projection's error when its check waits for the conversion."""
import ctypes as C

import numpy as np
import pytest

import oracle
from faust_amd import _lib, fact, factparams, proj

pytestmark = pytest.mark.gpu


def _near(rng, shape, bits):
    """Magnitudes 1 + i 2^-bits: they share every digit above the last ones."""
    i = rng.integers(0, 1 << 11, size=shape).astype(np.float64)
    return np.asfortranarray((1.0 + i * 2.0 ** -bits) * rng.choice([-1.0, 1.0], size=shape))


@pytest.mark.parametrize("case,k", [("normal", 1), ("normal", 40), ("normal", 16899), ("near20", 700), ("near40", 5000),
                                    ("near52", 900), ("ties", 3000), ("zeros", 400), ("tiny", 2000)])
def test_sp_selection(gpu, case, k):
    rng = np.random.default_rng(k)
    shape = (130, 130)
    if case == "normal":
        M = rng.standard_normal(shape)
    elif case.startswith("near"):
        M = _near(rng, shape, int(case[4:]))
    elif case == "ties":
        M = rng.integers(-3, 4, size=shape).astype(np.float64)
    elif case == "zeros":  # fewer nonzeros than k
        M = rng.standard_normal(shape) * (rng.random(shape) < 0.01)
    else:
        M = rng.standard_normal(shape) * 2.0 ** rng.integers(-1070, -1000, size=shape)
    M = np.asfortranarray(M)
    got = proj.sp(shape, k, normalized=case != "tiny")(M)
    assert np.array_equal(got, oracle.prox("sp", M, k, normalized=case != "tiny"))


@pytest.mark.parametrize("shape,k", [((33, 70), 33), ((33, 70), 40), ((70, 33), 40), ((65, 64), 64), ((20, 30), 30)])
def test_splincol_whole_lines(gpu, shape, k):
    M = np.asfortranarray(np.random.default_rng(k).standard_normal(shape))
    assert np.array_equal(proj.splincol(shape, k)(M), oracle.prox("splincol", M, k))


@pytest.mark.parametrize("fmt", ["dynamic", "sparse", "dense"])
@pytest.mark.parametrize("dims,names", [((65, 64, 130), ("sp", "spcol")), ((1, 63, 129, 70), ("splin", "sp", "splincol")),
                                        ((200, 17, 260), ("spcol", "splin"))])
def test_palm4msa_tile_edges(gpu, dims, names, fmt):
    rng = np.random.default_rng(sum(dims))
    A = np.asfortranarray(rng.standard_normal((dims[0], dims[-1])))
    cons, ocons = [], []
    for i, nm in enumerate(names):
        r, c = dims[i], dims[i + 1]
        k = {"sp": max(1, r * c // 9), "spcol": max(1, r // 4), "splin": max(1, c // 5), "splincol": 3}[nm]
        cons.append(factparams.ConstraintInt(nm, r, c, k))
        ocons.append((nm, k, r, c))
    p = factparams.ParamsPalm4MSA(cons, factparams.StoppingCriterion(num_its=5), factor_format=fmt)
    res = fact.palm4msa(A, p, ret_raw=True)
    ref = oracle.palm4msa(A, ocons, num_its=5, record_traj=True, factor_format=fmt)
    assert res.lam == ref.lam and res.kinds() == ref.kinds
    for a, b in zip(res.dense_factors(), ref.factors):
        assert np.array_equal(a, b)
    assert np.array_equal(res.traj, ref.traj)


@pytest.mark.parametrize("fmt", ["dynamic", "dense"])
def test_zero_projection_raises(gpu, fmt):
    cons = [factparams.ConstraintInt("sp", 40, 40, 80)] * 2
    p = factparams.ParamsPalm4MSA(cons, factparams.StoppingCriterion(num_its=3), factor_format=fmt)
    with pytest.raises(_lib.FaustHipError, match="norm is zero"):
        fact.palm4msa(np.zeros((40, 40)), p, ret_raw=True)


def test_empty_dot(gpu):
    out = C.c_double(5.0)
    _lib.check(gpu.fh_dot(_lib.FH_F64, None, None, 0, C.byref(out), None))
    assert out.value == 0.0
