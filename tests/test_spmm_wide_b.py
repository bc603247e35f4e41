"""A B beyond the 4 GiB that 32-bit gather offsets reach: block height 16 has no variant for it and refuses it, whatever form the
size of the problem would call for (refused before anything is launched)."""
import pytest

import shflbw_sparse_nn_amd as S
import workloads as P


@pytest.mark.gpu
@pytest.mark.parametrize("M,K,N", [(512, 1000, 2200000), (4096, 130, 16600000)])
def test_block_height_16_refuses(torch_gpu, M, K, N):
    torch = torch_gpu
    assert K * N * 2 > 2 ** 32
    w = P.upload_weight(P.make_weight(M, K, 16, 0.4, False, 3, integer=True))
    buf = torch.zeros(64, dtype=torch.float16, device="cuda")  # never touched: the initialisation fails
    with pytest.raises(Exception, match="4 GiB"):
        S.SpmmBlockwiseOp().initialize(w, N, buf.data_ptr(), buf.data_ptr())
