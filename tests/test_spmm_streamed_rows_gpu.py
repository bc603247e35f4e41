"""D of whole lines from 96 MB on is stored by streaming stores (result_store_mode): both sides of the rule, every block height
and role-split variant, with and without C, several times over the same buffers, against exact integer products."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [16, 32, 64, 128])
@pytest.mark.parametrize("M,N,residual", [(4096, 12352, False), (4096, 12352, True), (4096, 12224, False), (256, 196736, False)])
def test_streamed_rows(torch_gpu, V, M, N, residual):
    torch = torch_gpu
    K, per = 1200, 24
    X = M // V
    rng = np.random.default_rng(V + N)
    cols = np.stack([np.sort(rng.choice(K, per, replace=False)) for _ in range(X)])
    values = rng.integers(-4, 5, size=(X, per, V)).astype(np.float16)
    perm = rng.permutation(M).astype(np.int32)
    w = S.BlockwiseSpMatrix()
    w.set(M, K, V, 1, (np.arange(X + 1) * per).astype(np.int32), cols.reshape(-1).astype(np.int32), values.reshape(-1), perm)
    w.transform_and_sync_device()
    B = torch.from_numpy(rng.integers(-4, 5, size=(K, N)).astype(np.float16)).cuda()
    C = torch.from_numpy(rng.integers(-4, 5, size=(M, N)).astype(np.float16)).cuda() if residual else None
    dense = torch.zeros((M, K), dtype=torch.float32)
    rows = torch.from_numpy(perm.astype(np.int64)).reshape(X, V)
    for p in range(X):
        dense[rows[p][:, None], torch.from_numpy(cols[p])[None, :]] = torch.from_numpy(values[p].T.astype(np.float32))
    ref = dense.cuda() @ B.float() + (C.float() if residual else 0.0)  # sums of integers below 2^11: exact
    for variant in [-1] + [i for i, n in enumerate(S.spmm_variants(V)) if n.startswith("ws")]:
        D = torch.empty((M, N), dtype=torch.float16, device="cuda")
        op = S.SpmmBlockwiseOp(variant)
        op.initialize(w, N, B.data_ptr(), D.data_ptr(), C.data_ptr() if residual else None)
        for _ in range(2):
            D.fill_(float("nan"))
            op(torch.cuda.current_stream().cuda_stream)
            assert torch.equal(D.float(), ref), variant
