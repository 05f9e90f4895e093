"""Performance cases: the products (and the conversion) that a program using this
library runs, through the torch entry points.

Matrices are drawn on the GPU from a seed:
  uniform   every row takes `per_row` random columns (repeats merged)
  bernoulli every entry is kept with probability `density`
  powerlaw  row lengths follow P(L = k) ~ (k - shift)^-exponent on 1 .. cap, random columns
  ragged    row lengths spread evenly over lo .. hi, random columns
  rmat      R-MAT edges (2^scale vertices, `samples` edges, repeats merged)
Columns are sorted within a row, as CSR builders leave them, and values lie in
[-1, 1).  `entry` is the call that a program makes:
  auto, auto_hint  csrspmm_auto without and with the longest row
  naive, warp_per_row, warp_per_row_fp4, warp_per_row_smem,
  warp_per_row_smem_fp4  the five forwards (the staged ones with the longest row)
  out       csrspmm_spmm_out added to a copy of another matrix
  plan      a CsrSpmmPlan kept by the program
  sparse    csrspmm_sparse on a torch.sparse_csr tensor with int64 indices
  dense_to_csr  the conversion of a dense matrix
"""
import math

import torch

import torch_csrspmm

DEVICE = "cuda"


def listed():
    return [
        # A small graph with one narrow feature block: the latency of a call.
        dict(name="small", kind="uniform", M=1024, K=1024, per_row=10, N=32, entry="auto"),
        # The two larger shapes of the drop-in benchmark, a pruned dense layer at
        # 5% and at 10%, through the float4 forwards with alpha and beta given.
        dict(name="pruned-4k", kind="bernoulli", M=4096, K=4096, density=0.05, N=128,
             entry="warp_per_row_fp4", alpha=1.1, beta=0.5),
        dict(name="pruned-8k", kind="bernoulli", M=8192, K=4096, density=0.10, N=256,
             entry="warp_per_row_smem_fp4", alpha=1.1, beta=0.5),
        # Uniform sparse systems, B a little above one L2 and far above it.
        dict(name="uniform-16k", kind="uniform", M=16384, K=16384, per_row=82, N=128, entry="auto"),
        dict(name="uniform-64k", kind="uniform", M=65536, K=65536, per_row=66, N=256, entry="auto"),
        # Power-law rows up to 16384 nonzeros, B of 128 MiB.
        dict(name="powerlaw-256k", kind="powerlaw", M=262144, K=262144, exponent=1.5, shift=0.7,
             cap=16384, N=128, entry="auto"),
        # The same law on half the columns, multiplied again and again with one A.
        dict(name="powerlaw-plan", kind="powerlaw", M=131072, K=131072, exponent=1.5, shift=0.7,
             cap=16384, N=64, entry="plan"),
        # A program that keeps the first of the five forwards, on skewed rows.
        dict(name="naive-skewed", kind="powerlaw", M=65536, K=65536, exponent=1.5, shift=0.7,
             cap=4096, N=96, entry="naive"),
        # A residual update of an odd number of columns, rows of 0 to 300.
        dict(name="ragged-odd", kind="ragged", M=30011, K=20021, lo=0, hi=300, N=47, entry="out",
             alpha=0.75, beta=1.0),
        # A graph held as torch.sparse_csr (int64 indices), 100 features.
        dict(name="graph-csr", kind="rmat", scale=17, samples=1 << 21, N=100, entry="sparse"),
        # A large graph with wide features, the largest call.
        dict(name="graph-wide", kind="rmat", scale=20, samples=1 << 24, N=512, entry="auto"),
        # Pruned weights converted to CSR.
        dict(name="convert", kind="bernoulli", M=8192, K=8192, density=0.05, N=0, entry="dense_to_csr"),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _columns(rng):
    return rng.choice([_log(rng, 16, 512), 4 * _log(rng, 4, 128), 32 << rng.randrange(5)])


FORWARDS = ["warp_per_row", "warp_per_row_fp4", "warp_per_row_smem", "warp_per_row_smem_fp4"]


def draw(rng):
    kind = rng.choice(["uniform", "uniform", "bernoulli", "powerlaw", "ragged", "rmat", "convert"])
    if kind == "convert":
        return dict(kind="bernoulli", M=_log(rng, 512, 16384), K=_log(rng, 512, 8192),
                    density=rng.uniform(0.01, 0.3), N=0, entry="dense_to_csr")
    entry = rng.choice(["auto", "auto", "auto_hint", "out", "plan", "sparse", "naive"] + FORWARDS)
    case = dict(kind=kind, N=_columns(rng), entry=entry)
    if entry in FORWARDS or entry == "out":
        case.update(alpha=rng.uniform(0.5, 1.5), beta=rng.choice([0.0, 0.5, 1.0]))
    if kind == "uniform":
        case.update(M=_log(rng, 1024, 131072), K=_log(rng, 1024, 131072))
        case["per_row"] = _log(rng, 4, 128)
    elif kind == "bernoulli":
        case.update(M=_log(rng, 512, 8192), K=_log(rng, 512, 8192), N=min(case["N"], 256),
                    density=rng.uniform(0.01, 0.3))
    elif kind == "powerlaw":
        case.update(M=_log(rng, 16384, 262144), K=_log(rng, 16384, 262144), exponent=1.5, shift=0.7,
                    cap=1 << rng.randrange(10, 15), N=min(case["N"], 256))
    elif kind == "ragged":
        case.update(M=_log(rng, 1024, 65536), K=_log(rng, 1024, 65536), lo=0, hi=_log(rng, 16, 512))
    else:
        scale = rng.randrange(14, 20)
        case.update(scale=scale, samples=rng.choice([8, 16]) << scale)
    return case


def _rows(case):
    return 1 << case["scale"] if case["kind"] == "rmat" else case["M"]


def _cols(case):
    return 1 << case["scale"] if case["kind"] == "rmat" else case["K"]


RMAT = (0.57, 0.19, 0.19, 0.05)


def _law(case):
    k = torch.arange(1, case["cap"] + 1, dtype=torch.float64)
    w = (k - case["shift"]).pow(-case["exponent"])
    return w / w.sum()


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _csr(case, g):
    """(rowptr int32, colidx int32, values float32) on the GPU."""
    M, K = _rows(case), _cols(case)
    kind = case["kind"]

    def rand(*size):
        return torch.rand(*size, device=DEVICE, generator=g)

    if kind == "bernoulli":
        r, c = torch.nonzero(rand(M, K) < case["density"], as_tuple=True)
    else:
        if kind == "rmat":
            n = case["samples"]
            r = torch.zeros(n, dtype=torch.int64, device=DEVICE)
            c = torch.zeros(n, dtype=torch.int64, device=DEVICE)
            a, b, cc, _ = RMAT
            for _ in range(case["scale"]):
                u = rand(n)
                r = 2 * r + (u >= a + b)
                c = 2 * c + (((u >= a) & (u < a + b)) | (u >= a + b + cc))
        else:
            if kind == "uniform":
                lens = torch.full((M,), min(case["per_row"], K), device=DEVICE)
            else:
                # evenly spread quantiles in random order
                q = (torch.randperm(M, device=DEVICE, generator=g) + rand(M).double()) / M
                if kind == "powerlaw":
                    lens = 1 + torch.searchsorted(_law(case).cumsum(0).to(DEVICE), q)
                    lens.clamp_(max=min(case["cap"], K))
                else:
                    lens = case["lo"] + (q * (case["hi"] - case["lo"] + 1)).long()
                    lens.clamp_(max=min(case["hi"], K))
            r = torch.repeat_interleave(torch.arange(M, device=DEVICE), lens)
            c = torch.randint(K, (r.numel(),), device=DEVICE, generator=g)
        key = torch.unique(r * K + c)
        r, c = key // K, key % K
    rowptr = torch.zeros(M + 1, dtype=torch.int32, device=DEVICE)
    rowptr[1:] = torch.bincount(r, minlength=M).cumsum(0)
    vals = rand(r.numel()) * 2 - 1
    return rowptr, c.int(), vals


def _inputs(case, seed):
    g = _generator(seed)
    M, K, N = _rows(case), _cols(case), case["N"]
    if case["entry"] == "dense_to_csr":
        # pruned to a set share, so the counts are the same for every seed
        keep = torch.randperm(M * K, device=DEVICE, generator=g)[:round(M * K * case["density"])]
        v = torch.rand(keep.numel(), device=DEVICE, generator=g) * 2 - 1
        d = torch.zeros(M * K, device=DEVICE)
        d[keep] = v.masked_fill_(v == 0, 0.5)
        d = d.view(M, K)
        return dict(D=d)
    rowptr, colidx, vals = _csr(case, g)
    s = dict(rowptr=rowptr, colidx=colidx, vals=vals, K=K,
             B=torch.rand(K, N, device=DEVICE, generator=g) * 2 - 1)
    if case["entry"] == "out":
        s["X"] = torch.rand(M, N, device=DEVICE, generator=g) * 2 - 1
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    entry = case["entry"]
    s.update(entry=entry, alpha=case.get("alpha", 1.0), beta=case.get("beta", 0.0))
    if entry in ("auto_hint", "warp_per_row_smem", "warp_per_row_smem_fp4"):
        s["longest"] = int(s["rowptr"].diff().max())
    elif entry == "plan":
        s["plan"] = torch_csrspmm.CsrSpmmPlan(s["rowptr"], s["colidx"], s["vals"], s["K"], n_hint=case["N"])
    elif entry == "sparse":
        s["A"] = torch.sparse_csr_tensor(s["rowptr"].long(), s["colidx"].long(), s["vals"],
                                         size=(s["rowptr"].numel() - 1, s["K"]), check_invariants=False)
    return s


def run(s):
    entry = s["entry"]
    if entry == "dense_to_csr":
        return torch_csrspmm.dense_to_csr(s["D"])
    if entry == "plan":
        return s["plan"].spmm(s["B"], s["alpha"], s["beta"])
    if entry == "sparse":
        return torch_csrspmm.csrspmm_sparse(s["A"], s["B"], s["alpha"], s["beta"])
    a = (s["rowptr"], s["colidx"], s["vals"])
    if entry == "auto":
        return torch_csrspmm.csrspmm_auto(*a, s["B"], s["alpha"], s["beta"])
    if entry == "auto_hint":
        return torch_csrspmm.csrspmm_auto(*a, s["B"], s["alpha"], s["beta"], s["longest"])
    if entry == "out":
        return torch_csrspmm.csrspmm_spmm_out(*a, s["B"], s["X"].clone(), s["alpha"], s["beta"])
    forward = getattr(torch_csrspmm, "csrspmm_" + entry)
    if "longest" in s:
        return forward(*a, s["longest"], s["B"], s["alpha"], s["beta"])
    return forward(*a, s["B"], s["alpha"], s["beta"])


def _expected(case):
    """(nonzeros, distinct columns) of the case's matrix, as expected."""
    M, K = _rows(case), _cols(case)
    kind = case["kind"]
    if kind == "bernoulli":
        return M * K * case["density"], float(K)
    if kind == "rmat":
        n, s = case["scale"], case["samples"]
        a, b, c, d = RMAT

        def hit(p):
            return -math.expm1(s * math.log1p(-p))

        cols = sum(math.comb(n, j) * hit((a + c) ** (n - j) * (b + d) ** j) for j in range(n + 1))
        nnz = sum(math.comb(n, i) * math.comb(n - i, j) * math.comb(n - i - j, k) *
                  hit(a ** (n - i - j - k) * b ** i * c ** j * d ** k)
                  for i in range(n + 1) for j in range(n + 1 - i) for k in range(n + 1 - i - j))
        return nnz, cols

    def distinct(length):
        return -K * math.expm1(length * math.log1p(-1.0 / K))

    if kind == "uniform":
        nnz = M * distinct(min(case["per_row"], K))
    elif kind == "powerlaw":
        law = _law(case)
        lens = torch.arange(1, case["cap"] + 1, dtype=torch.float64).clamp(max=min(case["cap"], K))
        nnz = M * float((law * -torch.expm1(lens * math.log1p(-1.0 / K)) * K).sum())
    else:
        span = range(case["lo"], case["hi"] + 1)
        nnz = M * sum(distinct(min(x, K)) for x in span) / len(span)
    return nnz, distinct(nnz)


def work(case):
    M, K, N = _rows(case), _cols(case), case["N"]
    nnz, cols = _expected(case)
    if case["entry"] == "dense_to_csr":
        return dict(bytes=4 * M * K + 4 * (M + 1) + 8 * nnz, flops=0)
    index = 8 if case["entry"] == "sparse" else 4
    reads = index * (M + 1) + (index + 4) * nnz + 4 * cols * N
    prior = 4 * M * N if case["entry"] == "out" else 0
    return dict(bytes=reads + prior + 4 * M * N, flops=2 * nnz * N)


def tolerance(case):
    if case["entry"] == "dense_to_csr":
        return "exact"
    # Sums in 32 bits of up to 16384 products, in any order and any number of parts.  Against
    # 64 bits the listed and drawn cases measured up to 6.4e-7 (rel) and 3.0e-5 (max, on the
    # long rows of a skewed matrix, whose sums are far above the result's root mean square).
    return dict(rel=2.5e-6, max=1.2e-4)


def exact(case, seed):
    s = _inputs(case, seed)
    if case["entry"] == "dense_to_csr":
        r, c = torch.nonzero(s["D"], as_tuple=True)
        rowptr = torch.zeros(case["M"] + 1, dtype=torch.int32, device=DEVICE)
        rowptr[1:] = torch.bincount(r, minlength=case["M"]).cumsum(0)
        return rowptr, c.int(), s["D"][r, c]
    M = s["rowptr"].numel() - 1
    A = torch.sparse_csr_tensor(s["rowptr"], s["colidx"], s["vals"].double(), size=(M, s["K"]),
                                check_invariants=False)
    C = case.get("alpha", 1.0) * torch.sparse.mm(A, s["B"].double())
    if "X" in s:
        C += case.get("beta", 0.0) * s["X"].double()
    return C
