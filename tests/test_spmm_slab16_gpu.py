"""GPU parity of the slab form of the SpMM for block height 16 against the CPU oracle, integer operands, bit for bit: odd
batches and panels of less than a step, column tiles that end early, more column tiles than compute units, the fewest and the
most rows of B, many panels per wave, panels without a kept vector, a residual, non-finite rows of B."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S
from oracle import oracle as O
import workloads as P
from workloads import run_spmm

pytestmark = pytest.mark.gpu


def _slab():
    return [i for i, n in enumerate(S.spmm_variants(16)) if n.startswith("slab")][0]


def _check(torch, w, B, Cmat=None, alpha=1.0, beta=None):
    got = run_spmm(torch, w, B, Cmat=Cmat, alpha=alpha, beta=beta, variant=_slab())
    with np.errstate(invalid="ignore", over="ignore"):
        ref = O.float_to_half(P.spmm_oracle(w, B) if Cmat is None else P.spmm_oracle(w, B, Cmat, alpha, 1.0 if beta is None else beta))
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got[~nan].view(np.uint16), ref[~nan].view(np.uint16))


@pytest.mark.parametrize("M,N,K,d,permute", [
    (16, 8, 1, 1.0, True),
    (48, 72, 40, 0.7, True),
    (2048, 1000, 777, 0.1, False),
    (512, 520, 1128, 0.5, True),      # the most rows of B
    (256, 17000, 96, 0.5, True),      # more column tiles than compute units: workgroups refill the slab
    (33728, 136, 130, 0.05, True),    # more rows than the waves of 256 workgroups hold ids of in one column tile
    (4096, 4096, 500, 0.1, True),
])
def test_exact_shapes(torch_gpu, M, N, K, d, permute):
    _check(torch_gpu, P.make_weight(M, K, 16, d, permute, 17, integer=True), P.make_dense(K, N, 17, integer=True))


@pytest.mark.parametrize("N", [8, 328])
def test_empty_panels_residual_and_non_finite(torch_gpu, N):
    V, K, X = 16, 300, 40
    rng = np.random.default_rng(3)
    counts = rng.choice([0, 0, 1, 5, 16, 31, 33, 64, 65, 290], size=X)
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
