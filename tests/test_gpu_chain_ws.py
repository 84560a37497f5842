"""The workspace of chain products: the FP64 row-major form's room is asked for
only where the form can run, is never needed for a call to be accepted, and a
one-factor Faust shares none between streams, captured graphs or with the
allocation-free entry point."""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp
import torch

import faust_amd
import oracle
from faust_amd import _lib
from faust_amd.bsr import rand_bsr

pytestmark = pytest.mark.gpu


def _launches(F):
    n = C.c_int()
    _lib.check(_lib.lib().fh_faust_last_launches(F.h, C.byref(n)))
    return n.value


def _capture(call):
    """call() in a graph of its own, on a side stream that nothing has run on."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        g.capture_begin(capture_error_mode="thread_local")
        try:
            call()
        finally:
            g.capture_end()
    torch.cuda.current_stream().wait_stream(s)
    return g


def _replays_right(g, facs, op, X, Y):
    for _ in range(3):
        X.copy_(torch.randn(X.shape, dtype=X.dtype, device="cuda"))
        g.replay()
        torch.cuda.synchronize()
        want = oracle.chain_multiply(facs, np.asfortranarray(X.cpu().numpy().T), op)
        assert np.array_equal(Y.cpu().numpy().T, want)


@pytest.mark.parametrize("autotune", ["0", "1"])
@pytest.mark.parametrize("p", [12, 300])  # below and above the rule's line
def test_one_factor_captured_first(gpu, monkeypatch, p, autotune):
    monkeypatch.setenv("FH_AUTOTUNE", autotune)
    rng = np.random.default_rng(p)
    facs = [faust_amd.rand_csr(3001, 2501, 9, rng)]
    F, W = faust_amd.Faust(facs), faust_amd.Faust(facs)
    for G, V, op, n, m in ((F, W, "N", 2501, 3001), (F.T, W.T, "T", 3001, 2501)):
        X = torch.zeros((p, n), dtype=torch.float64, device="cuda")
        Y = torch.empty((p, m), dtype=torch.float64, device="cuda")
        V.matmul_device(X, Y)  # the kernels are loaded, the forms measured; G's handle has no workspace yet
        g = _capture(lambda: G.matmul_device(X, Y))
        assert _launches(G) == 1
        _replays_right(g, facs, op, X, Y)


def test_capture_keeps_to_the_room_there_is(gpu, monkeypatch):
    # a chain warmed up in the form that one launch per factor takes: the row-major one's room is not there
    monkeypatch.setenv("FH_AUTOTUNE", "0")
    rng = np.random.default_rng(2)
    facs = [faust_amd.rand_csr(3001, 3001, 9, rng) for _ in range(2)]
    F = faust_amd.Faust(facs)
    X = torch.randn((64, 3001), dtype=torch.float64, device="cuda")
    Y = torch.empty_like(X)
    monkeypatch.setenv("FH_CHAIN_FUSED", "0")
    F.matmul_device(X, Y)
    assert _launches(F) == 2
    monkeypatch.delenv("FH_CHAIN_FUSED")
    g = _capture(lambda: F.matmul_device(X, Y))
    assert _launches(F) == 2
    _replays_right(g, facs, "N", X, Y)
    F.matmul_device(X, Y)  # the graph holds the buffers: they stay where they are
    assert _launches(F) == 2
    _replays_right(g, facs, "N", X, Y)


@pytest.mark.parametrize("op", ["N", "T"])
def test_graph_keeps_its_workspace(gpu, monkeypatch, op):
    # fewer columns than the graph's, whose row-major form takes more room than the graph's intermediate
    monkeypatch.setenv("FH_AUTOTUNE", "0")
    rng = np.random.default_rng(3)
    dims = ((3001, 3001), (3001, 16001)) if op == "N" else ((16001, 3001), (3001, 3001))
    facs = [faust_amd.rand_csr(m, n, 9, rng) for m, n in dims]
    F = faust_amd.Faust(facs)
    X = torch.randn((400, 16001), dtype=torch.float64, device="cuda")
    Y = torch.empty((400, 3001), dtype=torch.float64, device="cuda")

    def multiply(p):  # F.T would be a handle of its own
        _lib.check(gpu.fh_faust_multiply(F.h, op.encode(), X.data_ptr(), p, Y.data_ptr(),
                                         torch.cuda.current_stream().cuda_stream))

    monkeypatch.setenv("FH_CHAIN_FUSED", "0")
    multiply(100)
    g = _capture(lambda: multiply(100))
    monkeypatch.delenv("FH_CHAIN_FUSED")
    for autotune in ("0", "1"):
        monkeypatch.setenv("FH_AUTOTUNE", autotune)
        multiply(64)
        assert _launches(F) == 2
        _replays_right(g, facs, op, X[:100], Y[:100])
    multiply(400)  # more columns need more room anyway
    assert _launches(F) == 3


def test_one_factor_on_two_streams(gpu, monkeypatch):
    # the copy of X belongs to the first stream; the second runs without it, and they overlap
    monkeypatch.setenv("FH_AUTOTUNE", "0")
    rng = np.random.default_rng(4)
    facs = [faust_amd.rand_csr(20001, 20001, 12, rng)]
    F = faust_amd.Faust(facs)
    Xs = [torch.randn((256, 20001), dtype=torch.float64, device="cuda") for _ in range(2)]
    Ys = [torch.empty_like(X) for X in Xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    seen = [set(), set()]
    for _ in range(8):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                F.matmul_device(Xs[i], Ys[i])
                seen[i].add(_launches(F))
    torch.cuda.synchronize()
    assert seen == [{2}, {1}]
    for X, Y in zip(Xs, Ys):
        assert np.array_equal(Y.cpu().numpy().T, oracle.chain_multiply(facs, np.asfortranarray(X.cpu().numpy().T), "N"))


def test_one_factor_noalloc_uses_no_scratch(gpu, monkeypatch):
    monkeypatch.setenv("FH_AUTOTUNE", "0")
    rng = np.random.default_rng(6)
    facs = [faust_amd.rand_csr(3001, 3001, 9, rng)]
    F = faust_amd.Faust(facs)
    X = torch.randn((64, 3001), dtype=torch.float64, device="cuda")
    Y = torch.empty_like(X)
    _lib.check(gpu.fh_faust_multiply_noalloc(F.h, b"N", C.c_void_p(X.data_ptr()), 64, C.c_void_p(Y.data_ptr()),
                                             C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert _launches(F) == 1
    assert np.array_equal(Y.cpu().numpy().T, oracle.chain_multiply(facs, np.asfortranarray(X.cpu().numpy().T), "N"))


@pytest.mark.parametrize("mode", ["per_factor", "short"])
def test_no_room_where_the_form_is_not_run(gpu, monkeypatch, mode):
    # 512 MB of X: a copy of it would show in the device's free memory
    monkeypatch.setenv("FH_AUTOTUNE", "0")
    rng = np.random.default_rng(7)
    n, p = (1 << 14, 1 << 12) if mode == "per_factor" else (1 << 10, 1 << 16)  # short: one-launch sizes
    facs = [faust_amd.rand_csr(n, n, 2, rng)] * (1 if mode == "per_factor" else 2)
    F = faust_amd.Faust(facs)
    if mode == "per_factor":
        _lib.check(gpu.fh_faust_set_mul_mode(F.h, 1))
    X = torch.ones((p, n), dtype=torch.float64, device="cuda")
    Y = torch.empty_like(X)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    F.matmul_device(X, Y)
    torch.cuda.synchronize()
    used = free - torch.cuda.mem_get_info()[0]
    base = 0 if mode == "per_factor" else 8 * n * p  # one column-major intermediate
    assert used < base + (256 << 20)


def test_fp32_capture_keeps_to_the_room_there_is(gpu):
    # 20 columns one way leave room for 36 the other way in plain columns, not in whole panels of 32
    rng = np.random.default_rng(9)
    facs = [rand_bsr(d[0], d[1], 32, 2, rng).astype(np.float32) for d in ((6400, 3200), (3200, 64))]
    F = faust_amd.Faust(facs, dtype=np.float32, act_dtype=np.float32)
    F.matmul_device(torch.randn((20, 64), device="cuda"))
    W = faust_amd.Faust(facs, dtype=np.float32, act_dtype=np.float32).T
    X = torch.randn((36, 6400), device="cuda")
    Y = torch.empty((36, 64), device="cuda")
    W.matmul_device(X, Y)

    def transposed():  # F.T would be a handle of its own
        _lib.check(gpu.fh_faust_multiply(F.h, b"T", X.data_ptr(), 36, Y.data_ptr(),
                                         torch.cuda.current_stream().cuda_stream))

    g = _capture(transposed)
    for _ in range(3):
        X.copy_(torch.randn(X.shape, device="cuda"))
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(Y, W.matmul_device(X))
        transposed()  # and the graph's buffers stay where they are


def _banded(n, per_row):
    """per_row entries (in turn) at consecutive columns around the diagonal."""
    k = np.resize(per_row, n)
    cols = np.concatenate([(np.arange(c) + min(max(i - c // 2, 0), n - c)) for i, c in enumerate(k)])
    data = np.random.default_rng(n).standard_normal(len(cols))
    return sp.csr_matrix((data, cols, np.concatenate([[0], np.cumsum(k)])), shape=(n, n))


def test_measured_form_is_of_the_row_widths(gpu, monkeypatch):
    # equal shapes and entries, rows of 7 (8 ELL slots) and of 3 and 11 (16 slots).  For banded factors the
    # unmeasured choice is one launch per factor, and the row-major form the quicker one at this size
    n, p = 8000, 250
    narrow, wide = [_banded(n, [7])] * 2, [_banded(n, [3, 11])] * 2
    A, B = faust_amd.Faust(narrow), faust_amd.Faust(wide)
    X = torch.randn((256, n), dtype=torch.float64, device="cuda")
    Y = torch.empty_like(X)
    _lib.check(gpu.fh_autotune_clear())
    monkeypatch.setenv("FH_AUTOTUNE", "1")
    A.matmul_device(X[:p], Y[:p])
    B.matmul_device(X, Y)  # B's handle has the form's room, its form for p columns is not measured
    assert _launches(A) == _launches(B) == 3
    g = _capture(lambda: B.matmul_device(X[:p], Y[:p]))
    assert _launches(B) == 2
    _replays_right(g, wide, "N", X[:p], Y[:p])


@pytest.mark.parametrize("op", ["N", "T"])
def test_unmeasured_form_is_of_the_locality(gpu, monkeypatch, op):
    # one launch per factor on column-major intermediates where a row's entries lie by those of the row before;
    # row-major intermediates for uniform ones of the same size
    monkeypatch.setenv("FH_AUTOTUNE", "0")
    n, p = 8000, 64
    for facs, launches in (([_banded(n, [7])] * 2, 2),
                           ([faust_amd.rand_csr(n, n, 7, np.random.default_rng(i)) for i in range(2)], 3)):
        F = faust_amd.Faust(facs)
        G = F if op == "N" else F.T
        X = torch.randn((p, n), dtype=torch.float64, device="cuda")
        Y = G.matmul_device(X)
        assert _launches(G) == launches
        want = oracle.chain_multiply(facs, np.asfortranarray(X.cpu().numpy().T), op)
        assert np.array_equal(Y.cpu().numpy().T, want)


def test_measured_form_is_of_the_locality(gpu, monkeypatch):
    # two entries in every row of both chains: banded ones keep one launch per factor, uniform ones are measured anew
    n, p = 16000, 64
    monkeypatch.setenv("FH_AUTOTUNE", "1")
    _lib.check(gpu.fh_autotune_clear())
    X = torch.randn((p, n), dtype=torch.float64, device="cuda")
    Y = torch.empty_like(X)
    for facs, launches in (([_banded(n, [2])] * 2, 2),
                           ([faust_amd.rand_csr(n, n, 2, np.random.default_rng(i)) for i in range(2)], 3)):
        F = faust_amd.Faust(facs)
        F.matmul_device(X, Y)
        assert _launches(F) == launches
