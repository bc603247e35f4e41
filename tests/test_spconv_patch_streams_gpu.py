"""Outputs of the patch form on both sides of its rule for streaming stores, filters that fill whole lines and that do not, one
workgroup and two per pixel, against exact integer products."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,W,C,F,V,permute", [
    (40, 56, 57, 16, 256, 64, True),    # 65 MB
    (40, 56, 53, 16, 256, 64, True),    # 61 MB: below 60 * 2^20
    (31, 61, 59, 24, 304, 16, True),    # 68 MB, pixels that start inside a line
    (37, 41, 43, 16, 640, 128, False),  # two workgroups per pixel, filters not permuted
])
def test_streamed_output(torch_gpu, B, H, W, C, F, V, permute):
    torch = torch_gpu
    per = 6
    X = F // V
    rng = np.random.default_rng(F + W)
    cols = np.stack([np.sort(rng.choice(C, per, replace=False)) for _ in range(X)])
    values = rng.integers(-4, 5, size=(X, per, V)).astype(np.float16)
    perm = rng.permutation(F).astype(np.int32) if permute else np.arange(F, dtype=np.int32)
    f = S.BlockwiseSpFilter()
    f.set(F, C, V, 1, (np.arange(X + 1) * per).astype(np.int32), cols.reshape(-1).astype(np.int32), values.reshape(-1),
          perm if permute else None, 1, 1, C)
    f.transform_and_sync_device()
    x = torch.from_numpy(rng.integers(-4, 5, size=(B, H, W, C)).astype(np.float16)).cuda()
    dense = torch.zeros((F, C), dtype=torch.float32)
    rows = torch.from_numpy(perm.astype(np.int64)).reshape(X, V)
    for p in range(X):
        dense[rows[p][:, None], torch.from_numpy(cols[p])[None, :]] = torch.from_numpy(values[p].T.astype(np.float32))
    ref = x.reshape(-1, C).float() @ dense.cuda().T  # sums of integers below 2^11: exact
    y = torch.empty((B * H * W, F), dtype=torch.float16, device="cuda")
    op = S.SpconvBlockwiseOp(5)
    op.initialize(f, B, H, W, 1, x.data_ptr(), y.data_ptr())
    for _ in range(2):
        y.fill_(float("nan"))
        op(torch.cuda.current_stream().cuda_stream)
        assert torch.equal(y.float(), ref)
