"""D whose rows do not start at whole lines is merged in the L2 where B, C and D are 80 MiB or more, under narrow tiles where D is 24 MiB
(result_store_mode): both sides of the rule, every block height, with and without C, rows and a base that start inside a line,
against exact integer products."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [16, 32, 64, 128])
@pytest.mark.parametrize("M,N,offset,residual", [
    (4096, 3080, 0, False),   # D of 25.2 MB, rows start inside a line: merged under narrow tiles
    (4096, 3080, 0, True),
    (4096, 2920, 0, False),   # 23.9 MB: written through
    (4096, 3136, 8, False),   # rows of whole lines from a base that is not at one
    (4096, 8008, 0, False),   # B and D 80.9 MiB: merged under all tiles
    (4096, 7912, 0, False),   # 79.9 MiB
    (4096, 8064, 8, False),
    (4096, 4616, 0, True),    # with C 82.7 MiB
    (256, 49160, 0, True),
])
def test_ragged_rows(torch_gpu, V, M, N, offset, residual):
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
        flat = torch.full((M * N + offset + 64,), float("nan"), dtype=torch.float16, device="cuda")
        op = S.SpmmBlockwiseOp(variant)
        op.initialize(w, N, B.data_ptr(), flat[offset:].data_ptr(), C.data_ptr() if residual else None)
        op(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(flat[offset:offset + M * N].reshape(M, N).float(), ref), variant
        assert torch.isnan(flat[:offset]).all() and torch.isnan(flat[offset + M * N:]).all()
