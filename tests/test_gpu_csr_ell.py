"""ELL views of FP64 CSR factors (pairs of slots, a lane per row) in the
one-launch chain and in the per-factor kernels, bit for bit against the
oracle: every stored width and one past the widest, rows with unused slots
and none, a last row without entries, both directions, and a dense operand
on either side.  Infinities stand against unused slots (column 0)."""
import numpy as np
import pytest
import scipy.sparse as sp

import faust_amd
import oracle

pytestmark = pytest.mark.gpu


def _factor(m, n, w, rng):
    """Rows of w, 1, 0 and w - 1 entries in turn (w in some row); columns cyclic, so a column's count is bounded too."""
    k = np.resize([w, 1, 0, w - 1], m)
    k[-1] = 0
    rows = np.repeat(np.arange(m), k)
    cols = np.concatenate([np.sort((i * 7 + np.arange(c)) % n) for i, c in enumerate(k)])
    return sp.csr_matrix((rng.standard_normal(len(rows)), (rows, cols)), shape=(m, n))


@pytest.mark.parametrize("form", ["chain", "factors"])
@pytest.mark.parametrize("w", [1, 2, 3, 4, 5, 8, 9, 16, 17, 24, 25, 32, 33])
def test_ell_bits(gpu, monkeypatch, w, form):
    monkeypatch.setenv("FH_AUTOTUNE", "0")
    if form == "factors":
        monkeypatch.setenv("FH_CHAIN_FUSED", "0")
        monkeypatch.setenv("FH_CHAIN_PF", "0")
    rng = np.random.default_rng(w)
    dims = (131, 257, 64, 190) if w > 2 else (1024, 1023, 64, 190)
    facs = [_factor(dims[i], dims[i + 1], min(w, dims[i + 1]), rng) for i in range(3)]
    F = faust_amd.Faust(facs)
    for p in (1, 5, 65):
        for G, op, n in ((F, "N", dims[-1]), (F.T, "T", dims[0])):
            X = np.asfortranarray(rng.standard_normal((n, p)))
            X[0, 0], X[-1, -1], X[n // 2, 0] = np.inf, -0.0, 1e308
            with np.errstate(invalid="ignore", over="ignore"):
                want = oracle.chain_multiply(facs, X, op)
            assert np.array_equal(G @ X, want, equal_nan=True)
