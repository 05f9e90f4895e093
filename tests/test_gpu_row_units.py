"""GPU parity of row units (Problem::row_units in rowgroup.hip): products whose
rows average 64 nonzeros or more, or about equal ones by the hint, give each
row of fewer than two segments to a group of its own and the segments of
longer rows to the segment blocks, a wave of which checks several slots.

Rows summed whole must equal the fp32 CSR-order restatement bit for bit, and
the split ones the combine's order: per call (summed in the main launch) and
through a stored plan (summed in the combine launch) all rows must agree bit
for bit.  Shapes: row counts that fill no block or group of XCDs, empty and
split rows next to each other, unsorted columns, more slots than waves
(several a wave), each group width, XCD slices (16384 x 128), column slices
one by one and in one launch, N = 1, odd and above one pass (600), and hints
(exact, with and without split rows; too small).
"""
import numpy as np
import pytest
import torch

import oracle
from csrspmm_amd import capi, gen
from csr_cases import csr_from_lengths, whole_row_limit

pytestmark = pytest.mark.gpu

TOL = 1e-5


def t(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


def check(C, rp, ci, va, B, C0, alpha, beta, whole, what):
    R, S = oracle.spmm_f64(rp, ci, va, B, C0, alpha, beta)
    bad, ratio, _, _ = oracle.check(C, R, S, TOL)
    assert bad == 0, f"{what}: {bad} elements off (max ratio {ratio:.3g})"
    F = oracle.spmm_f32_seq(rp, ci, va, B, C0, alpha, beta)
    rows = np.diff(rp) <= whole
    assert np.array_equal(C[rows], F[rows]), f"{what}: rows summed whole differ from the CSR order"


# (M, K, N, shortest, longest, split rows)
CASES = [
    (1, 70000, 64, 66000, 66000, ()),                      # one row, all of it split
    (33, 4096, 128, 2000, 4000, ()),                       # every row split
    (2101, 4096, 64, 600, 700, ()),                        # every row split, in row units
    (1003, 3000, 47, 0, 300, (0, 511, 512, 1002)),         # odd columns, no whole block
    (1003, 3000, 1, 0, 300, (5, 1002)),
    (2049, 2048, 8, 60, 140, (2048,)),
    (2049, 2048, 16, 60, 140, (0, 1)),
    (3001, 16384, 128, 40, 160, (7, 8, 9, 3000)),          # XCD slices
    (2500, 65536, 256, 0, 200, (100, 2499)),               # column slices, one launch each
    (9001, 4096, 256, 100, 180, (0, 4096, 9000)),          # more slots than segment waves
    (1500, 4096, 600, 0, 200, (3,)),
]


@pytest.mark.parametrize("algo", ["WarpPerRow", "WarpPerRowFp4", "WarpPerRowSmem", "WarpPerRowSmemFp4"])
@pytest.mark.parametrize("M,K,N,lo,hi,split", CASES)
def test_row_units(algo, M, K, N, lo, hi, split, gpu):
    rng = np.random.default_rng(M + N)
    lens = rng.integers(lo, hi + 1, size=M)
    lens[list(split)] = min(K, 1000)
    rp, ci, va = csr_from_lengths(lens, K, seed=N, unsorted_rows=(M // 2,))
    assert rp[-1] >= 64 * M
    B = gen.dense(N, gen.TAG_B, K, N)
    C0 = gen.dense(N, gen.TAG_C0, M, N)
    alpha, beta = (0.5, -1.5) if N % 2 == 0 else (1.0, 0.0)
    print(f"[row units] {algo} M={M} K={K} N={N} nnz={int(rp[-1])}", flush=True)
    args = (t(rp, gpu), t(ci, gpu), t(va, gpu))
    dB = t(B, gpu)
    dC = t(C0, gpu)
    capi.spmm(algo, *args, dB, dC, alpha, beta)
    torch.cuda.synchronize()
    C = dC.cpu().numpy()
    check(C, rp, ci, va, B, C0 if beta else None, alpha, beta, whole_row_limit(algo, rp, K, N), algo)
    plan = capi.Plan(algo, *args, K, n_hint=N)
    if plan.panelized_rows == 0:
        dC = t(C0, gpu)
        plan.spmm(dB, dC, alpha, beta)
        torch.cuda.synchronize()
        assert np.array_equal(C.view(np.uint32), dC.cpu().numpy().view(np.uint32)), \
            f"{algo}: per-call and stored-plan products differ"
    plan.close()


@pytest.mark.parametrize("algo,N", [("WarpPerRowFp4", 64), ("WarpPerRowSmemFp4", 256), ("WarpPerRow", 50),
                                    ("WarpPerRowSmem", 100)])
@pytest.mark.parametrize("lo,hi", [(20, 40), (150, 300), (300, 420)])
@pytest.mark.parametrize("given", ["longest", "too_small"])
def test_row_units_from_the_hint(algo, N, lo, hi, given, gpu):
    """About equal rows by the hint: below two segments no tables are built
    (every row whole).  A hint that is too small costs no correctness."""
    M, K = 40001, 5000  # enough items to be planned, B within the L2s
    rng = np.random.default_rng(hi)
    lens = rng.integers(lo, hi + 1, size=M)
    if given == "too_small":
        lens[[0, 77, M - 1]] = 1200
    rp, ci, va = csr_from_lengths(lens, K, seed=hi)
    B = gen.dense(N, gen.TAG_B, K, N)
    print(f"[row units] {algo} N={N} rows {lo}-{hi} hint {given}", flush=True)
    dC = torch.full((M, N), float("nan"), device=gpu)
    capi.spmm(algo, t(rp, gpu), t(ci, gpu), t(va, gpu), t(B, gpu), dC, 1.0, 0.0, hint=hi)
    torch.cuda.synchronize()
    whole = whole_row_limit(algo, rp, K, N, hi)
    check(dC.cpu().numpy(), rp, ci, va, B, None, 1.0, 0.0, whole, f"{algo} hint {hi}")
