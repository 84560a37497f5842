"""The LDS form of the power iteration (k_power_lds), bit for bit against the
oracle: one, two, four, eight and sixteen waves and the lengths around them,
rectangular chains, rows shorter than the operator's width, widths on both
sides of the register prefetch, dense operators, a chain that annihilates the
start vector's image, and shapes past the form's limits."""
import numpy as np
import pytest
import scipy.sparse as sp

import faust_amd
import oracle

pytestmark = pytest.mark.gpu


def _uneven(m, n, k, rng):
    """Rows of 1 .. k entries."""
    lens = 1 + np.arange(m) % k
    cols = np.concatenate([np.sort(rng.choice(n, size=c, replace=False)) for c in lens])
    return sp.csr_matrix((rng.standard_normal(len(cols)), cols, np.concatenate([[0], np.cumsum(lens)])), shape=(m, n))


@pytest.mark.parametrize("dims,k", [((1, 1), 1), ((63, 64), 2), ((64, 33, 64), 3), ((65, 64), 4), ((128, 70, 100), 5),
                                    ((129, 128), 6), ((200, 256), 9), ((257, 300), 2), ((512, 512, 500), 3),
                                    ((513, 700), 2), ((1000, 1024), 3), ((1024, 1025), 2)])
def test_power_lds_sparse_bits(gpu, dims, k):
    rng = np.random.default_rng(sum(dims))
    facs = [_uneven(dims[i], dims[i + 1], min(k, dims[i + 1]), rng) for i in range(len(dims) - 1)]
    for maxit in (1, 7, 100):
        got = faust_amd.Faust(facs).norm(2, max_num_its=maxit)
        assert got == oracle.spectral_norm(facs, maxit)[0]


@pytest.mark.parametrize("m,n", [(5, 9), (64, 64), (70, 64), (64, 70), (97, 90), (129, 128)])
def test_power_lds_dense_bits(gpu, m, n):
    rng = np.random.default_rng(m + n)
    facs = [np.asfortranarray(rng.standard_normal((m, n))), sp.csr_matrix(_uneven(n, n, 3, rng))]
    assert faust_amd.Faust(facs).norm(2) == oracle.spectral_norm(facs)[0]
    assert faust_amd.Faust(facs[:1]).norm(2) == oracle.spectral_norm(facs[:1])[0]


def test_power_lds_zero_product(gpu):
    # A B = 0 without either factor being zero
    a, b = np.zeros((40, 40)), np.zeros((40, 40))
    a[:, :20] = 1.0
    b[20:, :] = 1.0
    facs = [sp.csr_matrix(a), sp.csr_matrix(b)]
    assert faust_amd.Faust(facs).norm(2) == oracle.spectral_norm(facs)[0] == 0.0


@pytest.mark.parametrize("m,n", [(1, 5), (255, 257), (37, 1536), (1030, 1023), (1100, 2048), (2100, 260)])
def test_power_wide_dense_bits(gpu, monkeypatch, m, n):
    # k_pw_dense's parts and row groups, the boundary inside the first operator's launch and (2100) before it
    monkeypatch.setenv("FH_POWER_WIDE", "1")
    rng = np.random.default_rng(m)
    facs = [np.asfortranarray(rng.standard_normal((m, n))), _uneven(n, n, 4, rng)]
    for fs in (facs, facs[:1], facs[::-1] if m == n else facs[1:]):
        F = faust_amd.Faust(fs)
        for maxit in (1, 4, 5, 100):
            assert F.norm(2, max_num_its=maxit) == oracle.spectral_norm(fs, maxit)[0]
