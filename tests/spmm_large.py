"""Large SpMMs for the GPU tests: a weight of panels of several lengths against exact integer products, and the way that the library goes
about its launch."""
import os
import subprocess

import numpy as np

import shflbw_sparse_nn_amd as S

PLAN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin", "test_spmm_plan")


def lengths(X, per):
    """Kept vectors of the panels: long and short ones in turn, one that keeps nothing."""
    return [0 if p == X - 2 else per - (p % 3) * 40 if p % 2 else per + 30 for p in range(X)]


def launch(V, kept, K, N, permuted, residual):
    """(C is streamed, panels of the first half or 0) of the launch with the wide tiles of block height V"""
    args = [PLAN, "launch"] + [str(int(a)) for a in (V, K, N, permuted, residual)]
    out = subprocess.check_output(args, input=" ".join(map(str, kept)), text=True)
    return tuple(map(int, out.split()))


def check(torch, V, kept, K, N, permuted, residual):
    X = len(kept)
    M = V * X
    rng = np.random.default_rng(V + X + N)
    cols = [np.sort(rng.choice(K, n, replace=False)) for n in kept]
    values = [rng.integers(-1, 2, size=(n, V)).astype(np.float16) for n in kept]
    perm = rng.permutation(M).astype(np.int32) if permuted else None
    w = S.BlockwiseSpMatrix()
    w.set(M, K, V, 1, np.concatenate([[0], np.cumsum(kept)]).astype(np.int32), np.concatenate(cols).astype(np.int32),
          np.concatenate(values).reshape(-1), perm)
    w.transform_and_sync_device()
    B = torch.from_numpy(rng.integers(-1, 2, size=(K, N)).astype(np.float16)).cuda()
    C = torch.from_numpy(rng.integers(-4, 5, size=(M, N)).astype(np.float16)).cuda() if residual else None
    dense = torch.zeros((M, K), dtype=torch.float32)
    rows = torch.from_numpy((perm if permuted else np.arange(M)).astype(np.int64)).reshape(X, V)
    for p in range(X):
        dense[rows[p][:, None], torch.from_numpy(cols[p])[None, :]] = torch.from_numpy(values[p].T.astype(np.float32))
    ref = (dense.cuda() @ B.float()).half()  # sums of at most 3330 products of -1, 0 and 1, in practice below 2^11: exact
    assert float(ref.abs().max()) < 2000
    if residual:
        ref += C
    D = torch.empty((M, N), dtype=torch.float16, device="cuda")
    names = S.spmm_variants(V)
    for variant in [-1] + [i for i, n in enumerate(names) if n in ("ws128x64x4c4p_k32_s6", "ws64x128x4c4p_k32_s4")]:
        op = S.SpmmBlockwiseOp(variant)
        op.initialize(w, N, B.data_ptr(), D.data_ptr(), C.data_ptr() if residual else None)
        for _ in range(2):
            D.fill_(float("nan"))
            op(torch.cuda.current_stream().cuda_stream)
            assert torch.equal(D, ref), names[variant] if variant >= 0 else "the library's choice"
