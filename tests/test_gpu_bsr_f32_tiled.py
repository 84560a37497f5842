"""FP32 BSR chains with FP32 activations on tiled intermediates: the bits of the
per-wave kernel's column-major chain (FH_BSR_F32_KERNEL=0), for column counts
on both sides of a panel, a group and the form's lower limit, block rows of 0
to 9 blocks, both directions, graph replays, and the allocation-free entry
point with and without room for the tiles."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp
import torch

import faust_amd
from faust_amd import _lib

pytestmark = pytest.mark.gpu


def _bsr(nbr, nbc, rng, most=9):
    """Block rows of 0 .. most blocks in turn."""
    k = np.minimum(np.arange(nbr) % (most + 1), nbc)
    cols = np.concatenate([np.sort(rng.choice(nbc, size=c, replace=False)) for c in k])
    data = rng.standard_normal((int(k.sum()), 32, 32)).astype(np.float32)
    return sp.bsr_matrix((data, cols, np.concatenate([[0], np.cumsum(k)])), shape=(nbr * 32, nbc * 32))


@pytest.mark.parametrize("p", [1, 16, 17, 31, 32, 33, 127, 129, 300])
def test_tiled_chain_bits(gpu, monkeypatch, p):
    rng = np.random.default_rng(p)
    facs = [_bsr(12, 20, rng), _bsr(20, 9, rng), _bsr(9, 16, rng)]
    F = faust_amd.Faust(facs, dtype=np.float32, act_dtype=np.float32)
    for G, n in ((F, 16 * 32), (F.T, 12 * 32)):
        X = torch.randn((p, n), device="cuda").t()
        monkeypatch.delenv("FH_BSR_F32_KERNEL", raising=False)
        Y = G @ X
        monkeypatch.setenv("FH_BSR_F32_KERNEL", "0")
        assert torch.equal(Y, G @ X)


def test_tiled_chain_noalloc_and_graph(gpu, monkeypatch):
    rng = np.random.default_rng(1)
    F = faust_amd.Faust([_bsr(63, 63, rng, 3) for _ in range(2)], dtype=np.float32, act_dtype=np.float32)
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    # 4161 columns: one column-major intermediate of 2016 rows fits the 32 MiB scratch array, padded to 4192 it does not
    for p in (40, 4161):
        X = torch.randn((p, 2016), device="cuda")
        Y = torch.empty_like(X)
        _lib.check(gpu.fh_faust_multiply_noalloc(F.h, b"N", C.c_void_p(X.data_ptr()), p, C.c_void_p(Y.data_ptr()), st))
        assert torch.equal(Y, F.matmul_device(X))
    X = torch.randn((40, 2016), device="cuda")
    Y = F.matmul_device(X)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        F.matmul_device(X, Y)
    for _ in range(3):
        X.copy_(torch.randn(X.shape, device="cuda"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(Y, F.matmul_device(X))
