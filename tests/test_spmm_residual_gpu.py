"""GPU parity of D = A B + C where the pieces of C are loaded among the stages of a tile: tiles with fewer stages than
pieces and with many, several tiles per workgroup, a last column tile that ends inside a wave's share, panels without a
kept vector.  Integer operands, bit for bit against the CPU oracle, for every tile variant."""
import os
import subprocess
import sys

import numpy as np
import pytest

import shflbw_sparse_nn_amd as S
from oracle import oracle as O
import workloads as P
from workloads import run_spmm

pytestmark = pytest.mark.gpu


def _check(torch, w, N, variants, seed=5):
    B = P.make_dense(w["ncol"], N, seed, integer=True)
    C = P.make_dense(w["nrow"], N, seed, integer=True, stream=3)
    ref = O.float_to_half(P.spmm_oracle(w, B, C, 1.0, 1.0))
    for v in variants:
        print(S.spmm_variants(w["brow"])[v] if v >= 0 else "the library's choice", flush=True)
        got = run_spmm(torch, w, B, Cmat=C, variant=v)
        np.testing.assert_array_equal(got.view(np.uint16), ref.view(np.uint16))


@pytest.mark.parametrize("M,N,K,V,d", [
    (256, 8, 40, 16, 0.5), (256, 520, 600, 16, 0.3), (4096, 3080, 200, 16, 0.1),
    (256, 8, 40, 32, 0.5), (512, 1040, 700, 32, 0.5), (4096, 3080, 600, 32, 0.1),
    (256, 8, 40, 64, 0.5), (512, 1040, 700, 64, 0.5), (8192, 3080, 600, 64, 0.1),
    (256, 8, 40, 128, 0.5), (512, 1040, 700, 128, 0.5), (8192, 3080, 600, 128, 0.1),
])
def test_residual_all_variants(torch_gpu, M, N, K, V, d):
    w = P.make_weight(M, K, V, d, True, 13, integer=True)
    n = len(S.spmm_variants(V))
    _check(torch_gpu, w, N, [-1] + [v for v in range(n) if "slab" not in S.spmm_variants(V)[v] or K <= 1128])


@pytest.mark.parametrize("V", [16, 32, 64, 128])
def test_residual_empty_panels(torch_gpu, V):
    K, X = 300, 6
    counts = np.array([0, 33, 0, 5, 290, 0])
    rng = np.random.default_rng(3)
    w = dict(nrow=X * V, ncol=K, brow=V, bcol=1, nnzb=int(counts.sum()),
             indptr=np.concatenate([[0], np.cumsum(counts)]).astype(np.int32),
             indices=np.concatenate([np.sort(rng.choice(K, c, replace=False)) for c in counts]).astype(np.int32),
             values=rng.integers(-4, 5, size=int(counts.sum()) * V).astype(np.float16), row_permute_ids=O.row_permutation(X * V, 5))
    _check(torch_gpu, w, 776, range(-1, len(S.spmm_variants(V))))


_OTHER_BETA = """
import sys
import numpy as np, torch
import shflbw_sparse_nn_amd as S, workloads as P
from oracle import oracle as O
first, then = float(sys.argv[1]), float(sys.argv[2])
for V in (16, 32, 64, 128):
    w = P.make_weight(4 * V, 200, V, 0.4, True, 13, integer=True)
    B, C = P.make_dense(200, 72, 5, integer=True), P.make_dense(4 * V, 72, 5, integer=True, stream=3)
    ref = O.float_to_half(P.spmm_oracle(w, B, C, 1.0, then))
    m, dB, dC = P.upload_weight(w), P.to_dev(torch, B), P.to_dev(torch, C)
    for v, name in enumerate(S.spmm_variants(V)):
        D = torch.full((4 * V, 72), float("nan"), dtype=torch.float16, device="cuda")
        op = S.SpmmBlockwiseOp(v)
        st = op.initialize(m, 72, dB.data_ptr(), D.data_ptr(), dC.data_ptr(), 1.0, first)
        st.args.beta = then
        print(name, flush=True)
        op(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert np.array_equal(D.cpu().numpy().view(np.uint16), ref.view(np.uint16)), name
"""


@pytest.mark.parametrize("first,then", [("0", "1"), ("1", "0")])
def test_beta_of_a_state_may_change_after_init(torch_gpu, first, then):
    """beta and C are plain fields of the state: a caller may set another beta than the one the state was initialised with.
    In a process of its own, in which nothing has used the kernels of the other beta before."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    p = subprocess.run([sys.executable, "-c", _OTHER_BETA, first, then], cwd=root, stdout=subprocess.PIPE, stderr=subprocess.STDOUT,
                       text=True, timeout=100)
    print(p.stdout[-2000:], flush=True)
    assert p.returncode == 0, p.stdout[-2000:]
