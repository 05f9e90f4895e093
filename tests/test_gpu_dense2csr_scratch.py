"""Dense -> CSR that reads the matrix once (csrspmm_dense2csr_*_ex, through
torch_csrspmm.dense_to_csr): parts of up to 2048 columns, 512 a step, eight a
lane, whose kept values beyond three eighths do not fit the stage and are read
again.  Exact arrays against the oracle's host rule at the edges of lanes,
steps and parts, with more parts than one scan step takes, empty, full and
overflowing parts, and rows that start at any 4-byte address."""
import numpy as np
import pytest
import torch

import torch_csrspmm as tc
import oracle
from csrspmm_amd import capi

pytestmark = pytest.mark.gpu


def matrix(M, K, density, seed):
    rng = np.random.default_rng(seed)
    D = rng.uniform(-1, 1, (M, K)).astype(np.float32)
    D[rng.random((M, K)) > density] = 0.0
    D[0, :: max(1, K // 7)] = np.nan
    D[M - 1, K - 1] = np.inf
    D[M // 2] = 0.0                     # an empty row
    if M > 2:
        D[M // 3] = 1.0                 # a full one: its parts overflow the stage
    return D


def equal(got, want):
    for g, w in zip(got, want[:3]):
        g = g.cpu().numpy()
        assert g.dtype == w.dtype and np.array_equal(g.view(np.uint32), w.view(np.uint32))


@pytest.mark.parametrize("M,K,density,tol", [
    (1, 256, 0.5, 0.0), (3, 257, 0.3, 0.0), (9, 511, 0.05, 0.25), (9, 512, 0.36, 0.0), (9, 513, 0.4, 0.0),
    (7, 2047, 0.01, 0.0), (7, 2048, 0.3, 0.0), (7, 2049, 0.3, 0.0), (5, 4097, 0.6, 0.0), (5, 6151, 1.0, -1.0),
    (20001, 300, 0.02, 0.0), (6001, 4100, 0.01, 0.0),   # 20001 and 18003 parts: five scan blocks
    (140001, 256, 0.01, 0.0),                           # two steps a scan block
])
def test_read_once(M, K, density, tol, gpu):
    assert capi.hip().csrspmm_dense2csr_scratch_bytes(M, K) > 0
    D = matrix(M, K, density, M + K)
    want = oracle.dense2csr(D, tol)
    equal(tc.dense_to_csr(torch.from_numpy(D).to(gpu), tol), want)
    # rows of odd stride from an odd column on: 4-byte aligned only
    wide = torch.full((M, K + 2), 3.0, device=gpu)
    wide[:, 1:K + 1] = torch.from_numpy(D).to(gpu)
    equal(tc.dense_to_csr(wide[:, 1:K + 1], tol), want)


@pytest.mark.parametrize("K", [1, 255])
def test_few_columns_take_no_scratch(K, gpu):
    assert capi.hip().csrspmm_dense2csr_scratch_bytes(400, K) == 0
    D = matrix(400, K, 0.4, K)
    equal(tc.dense_to_csr(torch.from_numpy(D).to(gpu), 0.0), oracle.dense2csr(D, 0.0))


def test_scratch_is_checked(gpu):
    M, K = 64, 1000
    D = torch.from_numpy(matrix(M, K, 0.2, 5)).to(gpu)
    need = capi.hip().csrspmm_dense2csr_scratch_bytes(M, K)
    rowptr = torch.empty(M + 1, dtype=torch.int32, device=gpu)
    nnz = torch.empty(1, dtype=torch.int64, device=gpu)
    scratch = torch.empty(need + 256, dtype=torch.uint8, device=gpu)
    count = capi.hip().csrspmm_dense2csr_count_f32_ex
    args = (M, K, D.data_ptr(), K, 0.0, rowptr.data_ptr(), nnz.data_ptr())
    assert count(*args, scratch.data_ptr(), need - 1, None) == -5   # too small
    assert count(*args, scratch.data_ptr() + 4, need, None) == -1   # misaligned
    assert count(*args, scratch.data_ptr(), need, None) == 0
    torch.cuda.synchronize()
    assert int(nnz.item()) == int(rowptr[-1].item()) == oracle.dense2csr(D.cpu().numpy(), 0.0)[0][-1]
