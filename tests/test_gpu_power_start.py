"""The power iteration's start vector is right whatever was queued before the
process's first norm: a projection on another stream, not yet run, whose
scratch blocks (8 KiB each, the size of the start vector) the pool already
holds.  A start vector kept in one of them would be overwritten when the
projection runs.  One fresh process, since the vector is uploaded once."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SCRIPT = """
import ctypes as C
import numpy as np
import torch
import faust_amd
import oracle
from faust_amd import _lib

rng = np.random.default_rng(5)
facs = [faust_amd.rand_csr(200, 200, 3, rng) for _ in range(3)]
F = faust_amd.Faust(facs)
M = torch.sign(torch.randn((64, 64), dtype=torch.float64, device="cuda"))  # ties: the saved entries are used
want = oracle.prox("sp", np.asfortranarray(M.cpu().numpy().T), 1024, normalized=False)
A = torch.randn((4096, 4096), device="cuda")
torch.mm(A, A)
torch.cuda.synchronize()
s = torch.cuda.Stream()
with torch.cuda.stream(s):
    B = A
    for _ in range(60):  # some 60 ms of work ahead of the projection
        B = torch.mm(A, B)
    _lib.check(_lib.lib().fh_prox(_lib.FH_F64, 0, C.c_void_p(M.data_ptr()), 64, 64, 1024, 0, 0, None,
                                  C.c_void_p(s.cuda_stream)))
    got = F.norm(2, max_num_its=2)
torch.cuda.synchronize()
assert got == oracle.spectral_norm(facs, 2)[0]
assert F.norm(2, max_num_its=2) == got
assert np.array_equal(M.cpu().numpy().T, want)
print("start vector ok")
"""


def test_start_vector_outside_the_pool(gpu):
    r = subprocess.run([sys.executable, "-c", SCRIPT], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "start vector ok" in r.stdout, r.stdout + r.stderr
