"""The role-split kernels fetch rows of B through a descriptor that ends with B, and the padding slots of a panel have an offset
past that end.  Here B is as large as these kernels take (K * row bytes + row bytes just below 4 GiB), its last row is kept, and
its rows hold infinities wherever no kept vector reads them."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [16, 32, 64, 128])
def test_largest_b(torch_gpu, V):
    torch = torch_gpu
    K, N, M = 65535, 32760, 2 * V
    rng = np.random.default_rng(V)
    kept = [np.sort(np.append(rng.choice(K - 1, 36, replace=False), K - 1)), np.array([0, K - 1])]  # 37 and 2: padded to 64 slots
    values = rng.integers(-4, 5, size=(39, V)).astype(np.float16)
    w = S.BlockwiseSpMatrix()
    w.set(M, K, V, 1, np.array([0, 37, 39], np.int32), np.concatenate(kept).astype(np.int32), values.reshape(-1), None)
    w.transform_and_sync_device()
    B = torch.full((K, N), float("inf"), dtype=torch.float16, device="cuda")
    rows = np.unique(np.concatenate(kept))
    dense = torch.from_numpy(rng.integers(-4, 5, size=(len(rows), N)).astype(np.float16)).cuda()
    B[torch.from_numpy(rows).cuda()] = dense
    ref = np.zeros((M, N), np.float32)
    for p, (cols, v) in enumerate(((kept[0], values[:37]), (kept[1], values[37:]))):
        at = torch.from_numpy(np.searchsorted(rows, cols)).cuda()
        ref[p * V:(p + 1) * V] = (torch.from_numpy(v.astype(np.float32).T.copy()).cuda() @ dense[at].float()).cpu().numpy()
    for i, name in enumerate(S.spmm_variants(V)):
        if not name.startswith("ws"):
            continue
        print(name, flush=True)
        D = torch.full((M, N), float("nan"), dtype=torch.float16, device="cuda")
        op = S.SpmmBlockwiseOp(i)
        op.initialize(w, N, B.data_ptr(), D.data_ptr())
        op(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(D.cpu().numpy().astype(np.float32), ref, err_msg=name)
