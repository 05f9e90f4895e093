"""Naive with long rows relayed by a whole block (naive.hip relay_row): rows of
more than 512 nonzeros (more on larger products) are summed by the block's
four waves in turn, 32 nonzeros a turn, still one by one in CSR order, so every
row equals the fp32 restatement bit for bit.  Lengths around the limit, around
whole batches and whole rounds of batches, several long rows for one block
(blocks check rows an odd stride apart), empty rows, columns around a tile of
64, alpha and beta, and a B wide enough (4 GiB) for 64-bit row addresses."""
import numpy as np
import pytest
import torch

import torch_csrspmm as tc
import oracle
from csrspmm_amd import capi
from csr_cases import csr_from_lengths

pytestmark = pytest.mark.gpu

LENGTHS = [0, 511, 512, 513, 1, 543, 544, 545, 639, 640, 641, 767, 768, 769, 4096, 5000, 3, 0, 513]


def t(x, dev):
    return torch.from_numpy(np.ascontiguousarray(x)).to(dev)


@pytest.mark.parametrize("N", [1, 63, 64, 65, 130])
@pytest.mark.parametrize("rows", [1, 19, 200])
def test_relayed_rows(rows, N, gpu):
    K = 6000
    lens = np.resize(np.array(LENGTHS[::-1]), rows)
    lens[0] = 2000
    rp, ci, va = csr_from_lengths(lens, K, seed=N, unsorted_rows=(0,))
    rng = np.random.default_rng(rows)
    B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
    C0 = rng.uniform(-1, 1, (rows, N)).astype(np.float32)
    args = (t(rp, gpu), t(ci, gpu), t(va, gpu), t(B, gpu))
    print(f"[relay] rows={rows} N={N}", flush=True)
    C = tc.csrspmm_naive(*args, 1.0, 0.0).cpu().numpy()
    assert np.array_equal(C, oracle.spmm_f32_seq(rp, ci, va, B, None, 1.0, 0.0))
    dC = t(C0, gpu)
    capi.spmm("Naive", *args, dC, 0.5, -1.5)
    assert np.array_equal(dC.cpu().numpy(), oracle.spmm_f32_seq(rp, ci, va, B, C0, 0.5, -1.5))


def test_one_block_relays_many_rows(gpu):
    """All the long rows an odd stride apart: the ones that one block checks."""
    M, K, N = 1300, 3000, 32
    stride = (M + 63) // 64 | 1
    lens = np.full(M, 2)
    lens[5::stride] = 700
    rp, ci, va = csr_from_lengths(lens, K, seed=3)
    B = np.random.default_rng(4).uniform(-1, 1, (K, N)).astype(np.float32)
    C = tc.csrspmm_naive(t(rp, gpu), t(ci, gpu), t(va, gpu), t(B, gpu), 1.0, 0.0).cpu().numpy()
    assert np.array_equal(C, oracle.spmm_f32_seq(rp, ci, va, B, None, 1.0, 0.0))


@pytest.mark.parametrize("per_row", [35, 36, 600])
def test_fewer_blocks_on_a_large_b(per_row, gpu):
    """B just above 32 MiB around 36 nonzeros a row (blocks a CU are capped from
    there), without and with relayed rows."""
    M, K, N = 301, 70001, 120
    rp, ci, va = csr_from_lengths(np.full(M, per_row), K, seed=per_row)
    B = np.random.default_rng(9).uniform(-1, 1, (K, N)).astype(np.float32)
    C = tc.csrspmm_naive(t(rp, gpu), t(ci, gpu), t(va, gpu), t(B, gpu), 1.0, 0.0).cpu().numpy()
    assert np.array_equal(C, oracle.spmm_f32_seq(rp, ci, va, B, None, 1.0, 0.0))


def test_b_beyond_4_gib(gpu):
    """64-bit row addresses: a view of 70 columns of rows 2^17 floats apart."""
    K, N, ld = 9000, 70, 1 << 17
    wide = torch.empty((K, ld), device=gpu)
    B = np.random.default_rng(6).uniform(-1, 1, (K, N)).astype(np.float32)
    wide[:, :N] = t(B, gpu)
    lens = np.array([0, 3, 40, 513, 2000, 8999, 1])
    rp, ci, va = csr_from_lengths(lens, K, seed=8)
    C = tc.csrspmm_naive(t(rp, gpu), t(ci, gpu), t(va, gpu), wide[:, :N], 1.0, 0.0).cpu().numpy()
    assert np.array_equal(C, oracle.spmm_f32_seq(rp, ci, va, B, None, 1.0, 0.0))
