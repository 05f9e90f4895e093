"""csrspmm_sparse narrows both int64 index arrays in one launch: the same bits
as the int32 product, at sizes around a block, with no nonzeros and with views
as indices, and the errors of the arguments it refuses."""
import pytest
import torch

import torch_csrspmm as tc

pytestmark = [pytest.mark.gpu, pytest.mark.filterwarnings("ignore:Sparse CSR tensor support")]


def csr(M, K, per_row, dtype, dev):
    g = torch.Generator().manual_seed(M + per_row)
    rp = torch.arange(M + 1) * per_row
    ci = torch.rand(M, K, generator=g).argsort(1)[:, :per_row].sort(1).values.reshape(-1)
    va = torch.rand(M * per_row, generator=g) - 0.5
    return torch.sparse_csr_tensor(rp.to(dev, dtype), ci.to(dev, dtype), va.to(dev), size=(M, K))


@pytest.mark.parametrize("M,per_row", [(1, 1), (255, 1), (128, 3), (7, 0), (3000, 40)])
def test_index_types_agree(M, per_row, gpu):
    K, N = 200, 24
    B = torch.rand(K, N, device=gpu)
    got = tc.csrspmm_sparse(csr(M, K, per_row, torch.int64, gpu), B, 0.5, 2.0)
    A32 = csr(M, K, per_row, torch.int32, gpu)
    assert torch.equal(got, tc.csrspmm_sparse(A32, B, 0.5, 2.0))
    want = 0.5 * (A32.to_dense().double() @ B.double())
    assert (got.double() - want).abs().max() <= 1e-5


def test_refused(gpu):
    A = csr(5, 200, 2, torch.int64, gpu)
    B = torch.rand(200, 4, device=gpu)
    for a, b, match in [(A.to_dense(), B, "torch.sparse_csr"), (A, B[:-1], "B must be"),
                        (A, B[:, 0], "B must be"), (csr(5, 200, 2, torch.int64, "cpu"), B, "CUDA"),
                        (A.double(), B, "A_values must be float32"), (A, B.double(), "B must be float32")]:
        with pytest.raises(RuntimeError, match=match):
            tc.csrspmm_sparse(a, b)
    with pytest.raises(RuntimeError, match="unknown algorithm"):
        tc.csrspmm_sparse(A, B, algo="none")
