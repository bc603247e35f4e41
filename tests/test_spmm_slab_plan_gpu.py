"""The slab form's plan (slab_plan): chunks in one round and in several, jobs side by side by column tile and by chunk, D written
through, merged and streamed - each against exact integer products."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,M,K,N,per,residual", [
    (16, 33728, 777, 1000, 12, False),   # A larger than B: by chunk, parts of lines, written through (67 MB)
    (16, 33728, 777, 1304, 12, False),   # ... merged (88 MB, with B 86 MiB)
    (16, 20000, 1128, 136, 9, True),     # by chunk, written through; three column tiles, the last one of 8 columns
    (16, 8192, 384, 4096, 12, False),    # by tile, written through
    (16, 4096, 400, 12352, 5, False),    # by tile, streamed (101 MB)
    (32, 33792, 1100, 2104, 6, True),    # 33 tiles x 9 chunks at least: more jobs than compute units; merged
    (32, 33792, 500, 1600, 7, False),    # ... streamed
    (32, 1024, 1000, 2112, 200, False),  # one panel per wave
    (32, 64, 384, 20480, 3, False),      # more column tiles than compute units, two panels
])
def test_slab_plan(torch_gpu, V, M, K, N, per, residual):
    torch = torch_gpu
    X = M // V
    rng = np.random.default_rng(V + N)
    cols = np.stack([np.sort(rng.choice(K, per, replace=False)) for _ in range(X)])
    values = rng.integers(-2, 3, size=(X, per, V)).astype(np.float16)
    perm = rng.permutation(M).astype(np.int32)
    w = S.BlockwiseSpMatrix()
    w.set(M, K, V, 1, (np.arange(X + 1) * per).astype(np.int32), cols.reshape(-1).astype(np.int32), values.reshape(-1), perm)
    w.transform_and_sync_device()
    B = torch.from_numpy(rng.integers(-2, 3, size=(K, N)).astype(np.float16)).cuda()
    C = torch.from_numpy(rng.integers(-4, 5, size=(M, N)).astype(np.float16)).cuda() if residual else None
    dense = torch.zeros((M, K), dtype=torch.float32)
    rows = torch.from_numpy(perm.astype(np.int64)).reshape(X, V)
    for p in range(X):
        dense[rows[p][:, None], torch.from_numpy(cols[p])[None, :]] = torch.from_numpy(values[p].T.astype(np.float32))
    ref = dense.cuda() @ B.float() + (C.float() if residual else 0.0)  # sums of integers below 2^11: exact
    D = torch.empty((M, N), dtype=torch.float16, device="cuda")
    op = S.SpmmBlockwiseOp([i for i, n in enumerate(S.spmm_variants(V)) if n.startswith("slab")][0])
    op.initialize(w, N, B.data_ptr(), D.data_ptr(), C.data_ptr() if residual else None)
    for _ in range(2):
        D.fill_(float("nan"))
        op(torch.cuda.current_stream().cuda_stream)
        assert torch.equal(D.float(), ref)
