"""Kernels of the batched PALM4MSA engine at their edges: the sp selection by
candidates, the matrix-core GEMM tiles, the step sizes (rows past the
registers and past the LDS room; two rows per thread)."""
import numpy as np
import pytest

import faust_amd
import oracle
from faust_amd.batched import palm4msa_batched

pytestmark = pytest.mark.gpu


def _spread(n, rng):
    """Distinct magnitudes, neighbours a factor of exp(8 / n^2) apart (FP32 rounding does not reorder them)."""
    return rng.permutation(np.exp(np.linspace(0, 8, n * n))) * rng.choice([-1.0, 1.0], n * n)


def _target(kind, n, k, rng):
    a = _spread(n, rng)
    if kind == "thread":  # entries (t + 37 m) mod 1024 of every 1024, t = 0, are small: the list overflows
        m = np.arange(n * n // 1024)
        a[1024 * m + (37 * m) % 1024] *= 1e-6
    elif kind == "equal":
        a = np.sign(a)
    elif kind == "zeros":  # fewer nonzeros than k
        a[rng.permutation(n * n)[: n * n - k // 2]] = 0.0
    elif kind == "rows":
        a *= np.tile(np.where(np.arange(n) % 7 == 0, 1e3, 1.0), n)
    return np.asfortranarray(a.reshape(n, n, order="F"))


@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("kind,n,k", [("spread", 31, 5), ("spread", 32, 1), ("spread", 33, 1024), ("spread", 45, 1025),
                                      ("spread", 57, 3200), ("spread", 100, 2048), ("spread", 100, 2049),
                                      ("spread", 130, 4096), ("spread", 130, 4097), ("spread", 512, 2048),
                                      ("thread", 256, 900), ("equal", 90, 700), ("zeros", 90, 700), ("rows", 300, 1200),
                                      ("spread", 64, 4095), ("spread", 64, 4096)])
def test_sp_selection(gpu, kind, n, k, dtype):
    # factors start as 0 and the identity, so the first projection is the k largest entries of A (equal ones:
    # the lowest positions), divided by their norm
    A = _target(kind, n, k, np.random.default_rng(n + k))
    res = palm4msa_batched([A], 2, k=[k], dtype=dtype, num_its=1, refine_its=0)
    a = A.ravel(order="F")
    keep = np.argsort(-np.abs(a), kind="stable")[:k]
    want = np.zeros_like(a)
    want[keep] = a[keep]
    want /= np.linalg.norm(want)
    got = np.asarray(res.factors[0][0], dtype=np.float64).ravel(order="F")
    assert np.array_equal(got != 0, want != 0)
    # the gradient step is a rounded multiple of A, the norm a sum over 1024 threads of at most 64 + 10 roundings
    # for these sizes (512^2: 256 + 10): relative 2 (1 + 266 / 2 + 2) eps at the very most
    eps = np.finfo(np.float32 if dtype == "f32" else np.float64).eps
    assert np.max(np.abs(got - want)) <= 272 * eps * np.max(np.abs(want))


@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_gemm_tiles_same_bits(gpu, monkeypatch, dtype):
    rng = np.random.default_rng(4)
    As = [np.asfortranarray(rng.standard_normal((n, n))) for n in (1, 15, 64, 65, 97, 130, 200)]
    ks = [max(1, a.size // 2) for a in As]  # dense factors: every product is a GEMM
    res = {}
    for tile in ("32", "64", "65"):
        monkeypatch.setenv("FH_BGEMM_TILE", tile)
        r = palm4msa_batched(As, 3, k=ks, dtype=dtype, num_its=4, refine_its=1)
        res[tile] = [r.lambdas] + [np.asarray(f) for fs in r.factors for f in fs]
    for tile in ("32", "64"):
        for a, b in zip(res[tile], res["65"]):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("nf", [2, 3])
@pytest.mark.parametrize("per", [3, 16])
def test_power_rows_same_bits(gpu, monkeypatch, nf, per):
    # per = 16: the rows' ends of a 512 x 512 factor exceed the LDS room, and the factor that of the products
    rng = np.random.default_rng(nf + per)
    As = [np.asfortranarray(faust_amd.rand_csr(n, n, 8, rng).toarray() @ faust_amd.rand_csr(n, n, 8, rng).toarray()
                            * rng.exponential(1.0, (n, 1))) for n in (129, 300, 512)]
    res = []
    for reg in ("1", "0"):
        monkeypatch.setenv("FH_BATCH_POWER_REG", reg)
        r = palm4msa_batched(As, nf, k=[per * len(a) for a in As], dtype="f32", num_its=3, refine_its=0)
        res.append([r.lambdas] + [np.asarray(f) for fs in r.factors for f in fs])
    for a, b in zip(*res):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [3, 63, 257, 1030])
def test_dense_step_sizes(gpu, n):
    rng = np.random.default_rng(n)
    masks = [np.minimum((rng.random((n, n)) < 0.05) + np.eye(n), 1.0) for _ in range(2)]
    A = np.asfortranarray((masks[0] * rng.standard_normal((n, n))) @ (masks[1] * rng.standard_normal((n, n))))
    res = palm4msa_batched([A], 2, supports=[masks], dtype="f64", num_its=3, refine_its=0, warm_power=False)
    ref = oracle.palm4msa(A, [("supp", 0, n, n, True, False, masks[0]), ("supp", 0, n, n, True, False, masks[1])],
                          num_its=3)
    # as the neighbouring test of the same comparison: sums in another order, 1e-8
    assert abs(res.lambdas[0] - ref.lam) <= 1e-8 * abs(ref.lam)


def test_more_jobs_than_a_grid_dimension(gpu):
    # 33000 targets of two factors: 66000 targets and default factors to load
    rng = np.random.default_rng(33)
    As = [np.full((1, 1), v) for v in rng.standard_normal(33000)]
    kw = dict(dtype="f64", num_its=1, refine_its=0)
    got = palm4msa_batched(As, 2, k=[1] * len(As), **kw)
    ends = np.r_[0:40, 32960:33000]
    want = palm4msa_batched([As[i] for i in ends], 2, k=[1] * len(ends), **kw)
    assert np.array_equal(np.asarray(got.lambdas)[ends], want.lambdas)
    for i, fs in zip(ends, want.factors):
        assert all(np.array_equal(a, b) for a, b in zip(got.factors[i], fs))
