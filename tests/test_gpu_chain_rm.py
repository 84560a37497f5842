"""FP64 CSR chains on row-major intermediates (k_csr_rm_f64), bit for bit
against the oracle: panels and row blocks that end inside a tile, rows of 0,
1, 8, 9, 16, 17 and 40 entries, one factor, graph replays, and the
allocation-free entry point with and without room for the form."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

import faust_amd
import oracle

pytestmark = pytest.mark.gpu


def _launches(F):
    n = C.c_int()
    faust_amd._lib.check(faust_amd._lib.lib().fh_faust_last_launches(F.h, C.byref(n)))
    return n.value


def _ragged(m, n, rng):
    """Rows of 0, 1, 8, 9, 16, 17, 40 and 6 entries in turn."""
    k = np.resize([0, 1, 8, 9, 16, 17, 40, 6], m)
    indptr = np.concatenate([[0], np.cumsum(k)])
    cols = np.concatenate([np.sort(rng.choice(n, size=c, replace=False)) for c in k])
    return sp.csr_matrix((rng.standard_normal(len(cols)), cols, indptr), shape=(m, n))


@pytest.mark.parametrize("dims,p", [((1601, 2003, 1200), 257), ((1100, 1025), 224), ((2048, 1500, 1033, 1999), 96),
                                    ((6007, 5003), 31)])
def test_row_major_chain_bits(gpu, monkeypatch, dims, p):
    monkeypatch.setenv("FH_AUTOTUNE", "0")
    rng = np.random.default_rng(p)
    facs = [_ragged(dims[i], dims[i + 1], rng) for i in range(len(dims) - 1)]
    F = faust_amd.Faust(facs)
    for G, op, n in ((F, "N", dims[-1]), (F.T, "T", dims[0])):
        X = np.asfortranarray(rng.standard_normal((n, p)))
        X[rng.integers(0, n, 5), rng.integers(0, p, 5)] = [np.inf, -0.0, 0.0, 1e308, -np.inf]
        with np.errstate(invalid="ignore"):
            want = oracle.chain_multiply(facs, X, op)
        assert np.array_equal(G @ X, want, equal_nan=True)
        # terms: the densest factor's entries times the columns
        assert _launches(G) == (len(facs) + 1 if max(f.nnz for f in facs) * p >= 1 << 20 else len(facs))


def test_row_major_chain_noalloc_and_graph(gpu, monkeypatch):
    import torch
    monkeypatch.setenv("FH_AUTOTUNE", "0")
    rng = np.random.default_rng(3)
    facs = [faust_amd.rand_csr(3001, 3001, 9, rng) for _ in range(2)]
    F = faust_amd.Faust(facs)
    L = faust_amd._lib.lib()
    # 1000 columns: one intermediate fits the 32 MiB scratch array, X's row-major copy beside it does not
    for p, launches in ((64, 3), (1000, 2)):
        X = torch.randn((p, 3001), dtype=torch.float64, device="cuda")
        Y = torch.empty_like(X)
        st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        faust_amd._lib.check(L.fh_faust_multiply_noalloc(F.h, b"N", C.c_void_p(X.data_ptr()), p,
                                                         C.c_void_p(Y.data_ptr()), st))
        assert _launches(F) == launches
        want = oracle.chain_multiply(facs, np.asfortranarray(X.cpu().numpy().T), "N")
        assert np.array_equal(Y.cpu().numpy().T, want)
    X = torch.randn((64, 3001), dtype=torch.float64, device="cuda")
    Y = F.matmul_device(X)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        F.matmul_device(X, Y)
    for seed in range(3):
        X.copy_(torch.randn(X.shape, dtype=torch.float64, device="cuda"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(Y, F.matmul_device(X))
        assert np.array_equal(Y.cpu().numpy().T, oracle.chain_multiply(facs, np.asfortranarray(X.cpu().numpy().T), "N"))


@pytest.mark.parametrize("p", [1, 4, 31, 32, 33, 63, 256, 257])
@pytest.mark.parametrize("ell", ["1", "0"])
def test_fp32_panels(gpu, monkeypatch, p, ell):
    # FP32 CSR chains panel by panel: rows of 0 to 40 entries (CSR form) or up to 12 (ELL form); the same
    # bits from the two-rows-per-thread kernel, and close to FP64
    monkeypatch.setenv("FH_CSR_ELL", ell)
    rng = np.random.default_rng(p)
    dims = (333, 260, 129)
    facs = [_ragged(dims[i], dims[i + 1], rng) if ell == "0" else faust_amd.rand_csr(dims[i], dims[i + 1], 12, rng)
            for i in range(2)]
    F = faust_amd.Faust(facs, dtype=np.float32)
    for G, op, n in ((F, "N", dims[-1]), (F.T, "T", dims[0])):
        X = np.asfortranarray(rng.standard_normal((n, p)).astype(np.float32))
        monkeypatch.delenv("FH_CSR_RPT", raising=False)
        Y = G @ X
        monkeypatch.setenv("FH_CSR_RPT", "2")
        assert np.array_equal(Y, G @ X)
        f32 = [f.astype(np.float32).astype(np.float64) for f in facs]
        want = oracle.chain_multiply(f32, X.astype(np.float64), op)
        # two factors of at most 40 terms, each rounding below 2^-24 of the term sizes
        bound = np.abs(X.astype(np.float64))
        for f in (reversed(f32) if op == "N" else f32):
            bound = np.abs(f if op == "N" else f.T) @ bound
        assert np.all(np.abs(Y - want) <= 2.0 ** -24 * 2 * 41 * bound)
