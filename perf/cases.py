"""The calls whose speed is measured: Faust x dense products, dense products of
a Faust, PALM4MSA (single, hierarchical, batched) and the butterfly
factorization, through the package's public entry points.

A case is a dict of plain values.  `kind` picks the entry point:

  chain         F @ X (op N), F.T @ X (op T) or both, X a column-major CUDA
                tensor, as a program that keeps its data on the GPU calls it.
                form csr: factors of `nnz` entries per row at uniform columns;
                form bsr: 32 x 32 blocks, `nnz` blocks per block row.
                dtype f64 / f32 (CSR), bf16 (BF16 blocks and activations),
                f32_bf16 (FP32 blocks, BF16 activations), f32 (BSR: FP32 both)
  product       F.toarray() and F.norm(2) of an FP64 Faust
  palm          fact.palm4msa of one target
  hierarchical  fact.hierarchical of a Hadamard matrix with random signs
  batched       palm4msa_batched of many targets of mixed sizes
  butterfly     fact.butterfly of a CUDA matrix, applied to a block of columns
"""
import math

import numpy as np
import torch

import faust_amd
from faust_amd import Faust, fact, factparams
from faust_amd.batched import palm4msa_batched
from faust_amd.bsr import rand_bsr
from faust_amd.butterfly import support_csr


def listed():
    return [
        # one vector through a small operator: an iterative solver's matrix-free product (launch latency)
        dict(name="csr_f64_vector", kind="chain", form="csr", dtype="f64", rows=1024, inner=1024, cols=1024,
             factors=5, nnz=8, p=1, op="N"),
        # an operator and its adjoint on a block of vectors (the benchmark's chain_csr_f64 workload)
        dict(name="csr_f64_block", kind="chain", form="csr", dtype="f64", rows=1024, inner=1024, cols=1024,
             factors=5, nnz=8, p=64, op="NT"),
        # a larger rectangular operator and its adjoint, nothing a multiple of a tile
        dict(name="csr_f64_ragged", kind="chain", form="csr", dtype="f64", rows=6007, inner=5003, cols=4801,
             factors=4, nnz=7, p=250, op="NT"),
        # a large single-precision operator (the benchmark's chain_csr_f32 workload)
        dict(name="csr_f32_large", kind="chain", form="csr", dtype="f32", rows=16384, inner=16384, cols=16384,
             factors=6, nnz=12, p=256, op="N"),
        # block-sparse layers in serving precision (the benchmark's default workload)
        dict(name="bsr_bf16_large", kind="chain", form="bsr", dtype="bf16", rows=8192, inner=8192, cols=8192,
             factors=6, nnz=4, p=512, op="N"),
        # the same layers' transposes on a ragged batch, FP32 blocks kept
        dict(name="bsr_f32_bf16_ragged_t", kind="chain", form="bsr", dtype="f32_bf16", rows=4096, inner=4096,
             cols=4096, factors=4, nnz=5, p=201, op="T"),
        # block-sparse layers in FP32 throughout, the reference's MatBSR<float> precision
        dict(name="bsr_f32_large", kind="chain", form="bsr", dtype="f32", rows=8192, inner=8192, cols=8192,
             factors=6, nnz=4, p=512, op="N"),
        # densifying a Faust and its 2-norm (the benchmark's notebook workload)
        dict(name="product_dense", kind="product", form="dense", n=1024, factors=10, density=1.0),
        # one target factorized, all defaults but the iterations
        dict(name="palm_sp", kind="palm", n=256, factors=3, prox="sp", k=4, its=30, backend=2020),
        # fast-transform recovery, the reference's Hadamard demonstration
        dict(name="hierarchical_hadamard", kind="hierarchical", n=64, its=10),
        # many small factorizations together (the benchmark's palm workload, fewer targets and iterations)
        dict(name="palm_batched", kind="batched", targets=48, nmin=64, nmax=512, prox="sp", k=4, its=20),
        # closed-form butterfly factorization of a matrix on the GPU
        dict(name="butterfly_bbtree", kind="butterfly", n=4096, type="bbtree", perm="none", p=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["csr", "csr", "csr", "bsr", "bsr", "bsr", "product", "palm", "hierarchical", "batched",
                       "butterfly"])
    if kind == "csr":
        dtype = rng.choice(["f64", "f64", "f32"])
        hi = 6000 if dtype == "f64" else 16384
        inner = _log_int(rng, 200, hi)
        return dict(kind="chain", form="csr", dtype=dtype, rows=min(hi, max(64, int(inner * rng.uniform(0.7, 1.4)))),
                    inner=inner, cols=min(hi, max(64, int(inner * rng.uniform(0.7, 1.4)))),
                    factors=rng.randint(2, 6), nnz=rng.randint(2, 12), p=_log_int(rng, 1, 256),
                    op=rng.choice(["N", "T", "NT"]))
    if kind == "bsr":
        n = 32 * _log_int(rng, 16, 256)
        return dict(kind="chain", form="bsr", dtype=rng.choice(["bf16", "f32_bf16", "f32"]), rows=n, inner=n, cols=n,
                    factors=rng.randint(2, 6), nnz=rng.randint(2, 5), p=_log_int(rng, 1, 512),
                    op=rng.choice(["N", "T"]))
    if kind == "product":
        form = rng.choice(["dense", "sparse"])
        return dict(kind="product", form=form, n=_log_int(rng, 100, 1024), factors=rng.randint(3, 10),
                    density=1.0 if form == "dense" else rng.choice([0.02, 0.05, 0.2]))
    if kind == "palm":
        return dict(kind="palm", n=_log_int(rng, 32, 256), factors=rng.randint(2, 4),
                    prox=rng.choice(["sp", "splin", "spcol"]), k=rng.randint(3, 6), its=rng.randint(5, 30),
                    backend=rng.choice([2016, 2020, 2020]))
    if kind == "hierarchical":
        return dict(kind="hierarchical", n=rng.choice([16, 32, 64]), its=rng.randint(4, 10))
    if kind == "batched":
        prox = rng.choice(["sp", "sp", "supp"])
        lo, hi = rng.choice([(32, 100), (64, 256), (64, 512)])
        return dict(kind="batched", targets=_log_int(rng, 6, 48), nmin=lo, nmax=hi, prox=prox, k=rng.randint(3, 5),
                    its=rng.randint(5, 20))
    return dict(kind="butterfly", n=2 ** rng.randint(6, 12), type=rng.choice(["bbtree", "right", "left"]),
                perm=rng.choice(["none", "bitrev"]), p=_log_int(rng, 16, 128))


# ---------------------------------------------------------------- inputs
_ACT = {("csr", "f64"): torch.float64, ("csr", "f32"): torch.float32, ("bsr", "bf16"): torch.bfloat16,
        ("bsr", "f32_bf16"): torch.bfloat16, ("bsr", "f32"): torch.float32}


def _dims(case):
    return [case["rows"]] + [case["inner"]] * (case["factors"] - 1) + [case["cols"]]


def _chain_factors(case, seed):
    rng = np.random.default_rng(seed)
    d = _dims(case)
    if case["form"] == "csr":
        dt = np.float64 if case["dtype"] == "f64" else np.float32
        return [faust_amd.rand_csr(d[i], d[i + 1], min(case["nnz"], d[i + 1]), rng, dtype=dt)
                for i in range(len(d) - 1)]
    nb = min(case["nnz"], case["inner"] // 32)
    facs = [rand_bsr(d[i], d[i + 1], 32, nb, rng, scale=1 / math.sqrt(32 * nb)) for i in range(len(d) - 1)]
    if case["dtype"] == "bf16":  # the values the factors are stored in
        for f in facs:
            f.data = torch.from_numpy(f.data).to(torch.bfloat16).double().numpy()
        return facs
    return [f.astype(np.float32) for f in facs]


def _chain_x(case, seed, op):
    n = case["cols"] if op == "N" else case["rows"]
    g = torch.Generator(device="cuda").manual_seed(2 * int(seed) + (op == "T"))
    X = torch.randn((case["p"], n), generator=g, device="cuda", dtype=torch.float64)
    return X.to(_ACT[case["form"], case["dtype"]]).t()  # n x p, column-major


def _dense_factors(case, seed):
    """U(0, 1) factors, dense or with density * n entries per row, as pyfaust.rand makes them."""
    rng = np.random.default_rng(seed)
    n = case["n"]
    if case["form"] == "dense":
        return [np.asfortranarray(rng.random((n, n))) for _ in range(case["factors"])]
    k = max(1, int(case["density"] * n))
    return [faust_amd.rand_csr(n, n, k, rng, values="uniform") for _ in range(case["factors"])]


def _sparse_target(n, factors, k, rng):
    P = np.eye(n)
    for _ in range(factors):
        P = faust_amd.rand_csr(n, n, min(k, n), rng) @ P
    return np.asfortranarray(P + 1e-3 * rng.standard_normal((n, n)))


def _hadamard(case, seed):
    """The order-n Hadamard matrix with random row and column signs and a random scale."""
    rng = np.random.default_rng(seed)
    H = np.ones((1, 1))
    while H.shape[0] < case["n"]:
        H = np.block([[H, H], [H, -H]])
    s, t = rng.choice([-1.0, 1.0], size=(2, case["n"]))
    return np.asfortranarray(rng.uniform(0.5, 2.0) * s[:, None] * H * t[None, :])


def _batch_sizes(case):
    """Powers of two between nmin and nmax, and one odd size in eight targets; the same for every seed."""
    rng = np.random.default_rng([case["targets"], case["nmin"], case["nmax"]])
    pow2 = [n for n in (32, 64, 128, 256, 512) if case["nmin"] <= n <= case["nmax"]]
    return [int(rng.integers(case["nmin"], case["nmax"] + 1)) if i % 8 == 7 else int(rng.choice(pow2))
            for i in range(case["targets"])]


def _butterfly_input(case, seed):
    n = case["n"]
    g = torch.Generator(device="cuda").manual_seed(int(seed))
    A = torch.randn((n, n), generator=g, device="cuda", dtype=torch.float64)
    X = torch.randn((case["p"], n), generator=g, device="cuda", dtype=torch.float64).t()
    return A, X


# ---------------------------------------------------------------- the calls
def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case)
    if kind == "chain":
        facs = _chain_factors(case, seed)
        bf = case["dtype"] == "bf16"
        kw = dict(act_dtype=np.float32) if (case["form"], case["dtype"]) == ("bsr", "f32") else {}
        F = Faust(facs, dtype="bf16" if bf else np.float64 if case["dtype"] == "f64" else np.float32, **kw)
        s["calls"] = [(F if op == "N" else F.T, _chain_x(case, seed, op)) for op in case["op"]]
    elif kind == "product":
        s["F"] = Faust(_dense_factors(case, seed))
    elif kind == "palm":
        n, k = case["n"], case["k"]
        s["A"] = _sparse_target(n, case["factors"], k, np.random.default_rng(seed))
        value = k * n if case["prox"] == "sp" else k
        s["p"] = factparams.ParamsPalm4MSA([factparams.ConstraintInt(case["prox"], n, n, value)] * case["factors"],
                                           factparams.StoppingCriterion(num_its=case["its"]))
    elif kind == "hierarchical":
        s["A"] = _hadamard(case, seed)
        s["p"] = factparams.ParamsHierarchicalWHT(int(math.log2(case["n"])), num_its=case["its"])
    elif kind == "batched":
        rng = np.random.default_rng(seed)
        s["As"], s["kw"] = [], dict(dtype="f32", num_its=case["its"], refine_its=2)
        sizes = _batch_sizes(case)
        if case["prox"] == "sp":
            s["As"] = [_sparse_target(n, 3, case["k"], rng) for n in sizes]
            s["kw"]["k"] = [case["k"] * n for n in sizes]
        else:  # known supports, started near the factors: k butterfly factors of the largest power of two in each size
            s["kw"].update(supports=[], init=[], lambda_init=[])
            for n in sizes:
                n = 1 << (n.bit_length() - 1)
                masks = [support_csr(n, i % int(math.log2(n))).toarray() for i in range(3)]
                true = [m * rng.standard_normal((n, n)) for m in masks]
                s["As"].append(true[0] @ true[1] @ true[2])
                near = [m * (t + 0.1 * rng.standard_normal((n, n))) for m, t in zip(masks, true)]
                s["kw"]["supports"].append(masks)
                s["kw"]["init"].append([f / np.linalg.norm(f) for f in near])
                s["kw"]["lambda_init"].append(float(np.prod([np.linalg.norm(f) for f in near])))
    else:
        s["A"], s["X"] = _butterfly_input(case, seed)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "chain":
        return [F @ X for F, X in s["calls"]]
    if kind == "product":
        return {"product": s["F"].toarray(), "norm2": s["F"].norm(2)}
    if kind == "palm":
        F, lam = fact.palm4msa(s["A"], s["p"], ret_lambda=True, backend=case["backend"])
        return {"factors": [F.factors(i) for i in range(len(F))], "lambda": lam}
    if kind == "hierarchical":
        F, lam = fact.hierarchical(s["A"], s["p"], ret_lambda=True)
        return {"factors": [F.factors(i) for i in range(len(F))], "lambda": lam, "product": F.toarray()}
    if kind == "batched":
        r = palm4msa_batched(s["As"], 3, **s["kw"])
        return {"factors": [np.concatenate([fs[j].ravel(order="K") for fs in r.factors]) for j in range(3)],
                "lambda": r.lambdas, "relerr": r.relerr}
    F = fact.butterfly(s["A"], type=case["type"], perm=None if case["perm"] == "none" else case["perm"])
    return F @ s["X"]


# ---------------------------------------------------------------- what they cost at least, and how exact they are
def work(case):
    """Inputs and outputs once each, and the multiplications of the cheapest form of the same algorithm."""
    kind = case["kind"]
    if kind == "chain":
        d = _dims(case)
        if case["form"] == "csr":
            v = 8 if case["dtype"] == "f64" else 4
            a = v
            entries = [r * min(case["nnz"], c) for r, c in zip(d, d[1:])]
            fac = sum(e * (v + 4) + 4 * (r + 1) for e, r in zip(entries, d))
        else:
            v = 2 if case["dtype"] == "bf16" else 4
            a = 4 if case["dtype"] == "f32" else 2
            nb = min(case["nnz"], case["inner"] // 32)
            entries = [r * nb * 32 for r in d[:-1]]
            fac = sum(e * v + e // 256 for e in entries)
        per_call = fac + a * case["p"] * (d[0] + d[-1])
        return {"bytes": len(case["op"]) * per_call, "flops": len(case["op"]) * 2 * case["p"] * sum(entries)}
    if kind == "product":
        n, J = case["n"], case["factors"]
        nnz = n * n if case["form"] == "dense" else n * max(1, int(case["density"] * n))
        per = 8 if case["form"] == "dense" else 12
        return {"bytes": J * nnz * per + 8 * n * n, "flops": 2 * (J - 1) * nnz * n + 100 * 4 * J * nnz}
    if kind == "palm":  # per factor update: the error's product with each side, and its sparse x dense products
        n, J = case["n"], case["factors"]
        return {"bytes": 8 * n * n * (1 + J), "flops": case["its"] * J * (4 * n ** 3 + 4 * case["k"] * n * n)}
    if kind == "hierarchical":  # per level: a 2-factor PALM4MSA and one of all factors so far
        n, L = case["n"], int(math.log2(case["n"]))
        updates = case["its"] * sum(2 + (i + 2) for i in range(L - 1))
        return {"bytes": 8 * n * n * 2, "flops": updates * 4 * n ** 3}
    if kind == "batched":
        sizes = _batch_sizes(case)
        return {"bytes": sum(8 * n * n * 4 for n in sizes),
                "flops": sum(case["its"] * 3 * (4 * n ** 3 + 4 * case["k"] * n * n) for n in sizes)}
    n = case["n"]
    L = int(math.log2(n))
    out = 2 * n * 12 * L if case["type"] == "bbtree" else 8 * n * n * L
    return {"bytes": 8 * n * n + out + 16 * n * case["p"], "flops": 4 * n * n * L}


def tolerance(case):
    """About four times what exact(), other orders of the sums or inputs moved by 1e-15 show."""
    kind = case["kind"]
    if kind == "chain":
        if case["dtype"] == "f64":
            return {"rel": 2e-15}
        if case["dtype"] == "f32":
            return {"rel": 8e-7 if case["form"] == "csr" else 2e-6}
        return {"rel": 1.6e-2, "max": 0.1}
    if kind == "product":
        return {"rel": 5e-15}
    if kind in ("palm", "hierarchical"):
        return {"rel": 1e-14}
    if kind == "batched":  # FP32 sums in another order: 2e-7, unless one of them moves an entry across the sp threshold
        return {"rel": 1e-2, "max": 0.99} if case["prox"] == "sp" else {"rel": 1e-6}
    return {"rel": 1e-11}


def _tree(leaves):
    """Split points of the balanced tree over `leaves` factors: leading factors paired, then halved."""
    half = 1 << (math.ceil(math.log2(leaves)) - 1)
    pairs = leaves - half
    groups = [(2 * i, 2 * i + 2) for i in range(pairs)] + [(2 * pairs + i, 2 * pairs + i + 1)
                                                           for i in range(half - pairs)]
    return {(a, b): groups[len(groups) // 2][0] for groups in _halves(groups)
            for a, b in [(groups[0][0], groups[-1][1])]} | {(a, b): a + 1 for a, b in groups if b - a == 2}


def _halves(groups):
    if len(groups) > 1:
        yield groups
        yield from _halves(groups[:len(groups) // 2])
        yield from _halves(groups[len(groups) // 2:])


def _butterfly_leaves(A, type):
    """The (n, 2) row values of each butterfly factor of A: every split takes the best rank-1 block (FP64 SVD)."""
    n = A.shape[0]
    L = int(math.log2(n))
    tree = _tree(L)
    t = torch.arange(n)

    def field(i, at, bits, value):  # i with its bits [at, at + bits) replaced
        return (i & ~(((1 << bits) - 1) << at)) | (value << at)

    def split(V, a, b):
        if b - a == 1:
            return [V]
        c = {"bbtree": tree.get((a, b)), "right": a + 1, "left": b - 1}[type]
        bx, sx, by, sy = c - a, L - c, b - c, L - b
        rows = field(t[:, None], sx, bx, torch.arange(1 << bx)[None, :])
        cols = field(t[:, None], sy, by, torch.arange(1 << by)[None, :])
        block = V[rows[:, :, None], ((cols >> sy) & ((1 << (b - a)) - 1))[:, None, :]]
        U, S, Wt = torch.linalg.svd(block, full_matrices=False)
        r = S[:, :1].sqrt()
        X = torch.empty((n, 1 << bx), dtype=V.dtype)
        X[rows, ((t >> sx) & ((1 << bx) - 1))[:, None].expand_as(rows)] = U[:, :, 0] * r
        return split(X, a, c) + split(Wt[:, 0, :] * r, c, b)

    return split(A, 0, L)


def _butterfly_exact(case, seed):
    A, X = (x.cpu() for x in _butterfly_input(case, seed))
    n = case["n"]
    L = int(math.log2(n))
    r = torch.arange(n)
    if case["perm"] == "bitrev":  # A P^T is factorized and P put back
        rev = sum(((r >> b) & 1) << (L - 1 - b) for b in range(L))
        A, X = A[:, rev], X[rev]
    Y = X
    for i, V in reversed(list(enumerate(_butterfly_leaves(A, case["type"])))):
        s = 1 << (L - 1 - i)
        c0 = r & ~s
        Y = V[:, :1] * Y[c0] + V[:, 1:] * Y[c0 + s]
    return Y.numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "chain":
        out = []
        facs = [f.astype(np.float64) for f in _chain_factors(case, seed)]
        for op in case["op"]:
            Y = _chain_x(case, seed, op).double().cpu().numpy()
            for f in (reversed(facs) if op == "N" else facs):
                Y = (f if op == "N" else f.T) @ Y
            out.append(np.asarray(Y))
        return out
    if kind == "product":
        facs = [torch.from_numpy(np.asarray(f if case["form"] == "dense" else f.toarray())).cuda()
                for f in _dense_factors(case, seed)]
        P = facs[0]
        for f in facs[1:]:
            P = P @ f
        return {"product": P.cpu().numpy(), "norm2": float(torch.linalg.matrix_norm(P, 2))}
    if kind == "hierarchical":  # the factors are one choice of many; their product is the matrix
        return {"factors": None, "lambda": None, "product": _hadamard(case, seed)}
    if kind == "butterfly":
        return _butterfly_exact(case, seed)
    return None  # the end of a fixed number of iterations of a non-convex search has no other value
