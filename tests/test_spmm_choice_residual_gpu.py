"""The library's choice of the SpMM variant weighs what a C term costs each of them (spmm_estimate): shapes where it is another
one with C than without, both against the CPU oracle, integer operands, bit for bit."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S
from oracle import oracle as O
import workloads as P
from workloads import run_spmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,V,d", [
    (1680, 309, 13416, 16, 0.032), (3968, 1700, 1336, 32, 0.134), (26496, 2069, 384, 64, 0.087), (9472, 167, 4104, 128, 0.196),
])
def test_choice_with_and_without_c(torch_gpu, M, K, N, V, d):
    torch = torch_gpu
    w = P.make_weight(M, K, V, d, True, 13, integer=True)
    B, C = P.make_dense(K, N, 5, integer=True), P.make_dense(M, N, 5, integer=True, stream=3)
    mat = P.upload_weight(w)
    b, c, out = (torch.empty((r, N), dtype=torch.float16, device="cuda") for r in (K, M, M))
    plain = S.SpmmBlockwiseOp().initialize(mat, N, b.data_ptr(), out.data_ptr()).variant
    added = S.SpmmBlockwiseOp().initialize(mat, N, b.data_ptr(), out.data_ptr(), c.data_ptr()).variant
    assert plain != added
    for x, beta in ((None, 0.0), (C, 1.0)):
        ref = O.float_to_half(P.spmm_oracle(w, B, x, 1.0, beta))
        got = run_spmm(torch, w, B, Cmat=x, variant=-1)
        np.testing.assert_array_equal(got.view(np.uint16), ref.view(np.uint16))
