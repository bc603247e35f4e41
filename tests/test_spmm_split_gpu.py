"""GPU parity of the split form of the SpMM (few columns, the waves of a workgroup split the kept vectors) against the CPU
oracle, integer operands, bit for bit.  The shapes sit where it can go wrong: fewer steps than waves, a share of one step and
of many, the last column block partly and hardly used, one and two column blocks and several column tiles, row blocks that
do not fill the eight XCDs, panels without a kept vector, the row of zeros behind padding slots."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S
from oracle import oracle as O
import workloads as P
from workloads import run_spmm

pytestmark = pytest.mark.gpu


def _variant(V):
    return [i for i, n in enumerate(S.spmm_variants(V)) if n.startswith("split")][0]


def _check(torch, w, B, Cmat=None, alpha=1.0, beta=None, variant=None):
    got = run_spmm(torch, w, B, Cmat=Cmat, alpha=alpha, beta=beta, variant=_variant(w["brow"]) if variant is None else variant)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = O.float_to_half(P.spmm_oracle(w, B) if Cmat is None else P.spmm_oracle(w, B, Cmat, alpha, 1.0 if beta is None else beta))
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got[~nan].view(np.uint16), ref[~nan].view(np.uint16))


@pytest.mark.parametrize("V", [16, 32, 64, 128])
@pytest.mark.parametrize("M,N,K,d,permute", [
    (128, 8, 16, 1.0, True),      # one step
    (384, 24, 77, 0.5, True),     # fewer steps than waves, three columns of pieces
    (1152, 32, 1000, 0.1, False),
    (512, 40, 1500, 0.4, True),   # two column blocks, the second with eight columns
    (128, 64, 4096, 0.9, True),   # many steps per wave
    (640, 72, 333, 0.3, True),    # two column tiles, the second with eight columns
    (8448, 16, 200, 0.2, True),   # more workgroups than compute units
    (4096, 64, 520, 0.3, True),
])
def test_exact_shapes(torch_gpu, V, M, N, K, d, permute):
    _check(torch_gpu, P.make_weight(M, K, V, d, permute, 11, integer=True), P.make_dense(K, N, 11, integer=True))


@pytest.mark.parametrize("V", [16, 32, 64, 128])
@pytest.mark.parametrize("N", [8, 56])
def test_empty_panels_residual_and_non_finite(torch_gpu, V, N):
    K, X = 300, 6
    counts = np.array([0, 33, 0, 5, 290, 0])
    rng = np.random.default_rng(3)
    w = dict(nrow=X * V, ncol=K, brow=V, bcol=1, nnzb=int(counts.sum()),
             indptr=np.concatenate([[0], np.cumsum(counts)]).astype(np.int32),
             indices=np.concatenate([np.sort(rng.choice(K, c, replace=False)) for c in counts]).astype(np.int32),
             values=rng.integers(1, 5, size=int(counts.sum()) * V).astype(np.float16),  # no zero: 0 * inf is NaN in the oracle too
             row_permute_ids=O.row_permutation(X * V, 5))
    B = P.make_dense(K, N, 4, integer=True)
    C = P.make_dense(X * V, N, 4, integer=True, stream=3)
    _check(torch_gpu, w, B)
    _check(torch_gpu, w, B, C)
    _check(torch_gpu, w, B, C, alpha=2.0, beta=-0.5)
    B[0, 3], B[17, 7], B[299, 0] = np.inf, np.nan, -np.inf
    _check(torch_gpu, w, B)
