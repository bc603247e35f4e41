"""The library's choice of the SpMM variant (auto_spmm_variant).  With a C term it weighs what that costs each variant: shapes where the
fastest variant without C was measured 1.16 times and more the time of another one with it, results with and without C
against the CPU oracle, integer operands, bit for bit.  And shapes where rules of earlier versions took a variant of 1.12 to 1.45 times
the time of another (initialisation only)."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S
from oracle import oracle as O
import workloads as P
from workloads import run_spmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N,V,d,slow", [
    (1680, 309, 13416, 16, 0.032, None), (3968, 1700, 1336, 32, 0.134, None), (26496, 2069, 384, 64, 0.087, None),
    (9472, 167, 4104, 128, 0.196, None),
    (816, 168, 8368, 16, 0.221, "slab16x64"),                   # 11.9 us, fastest 9.0
    (704, 2844, 4288, 32, 0.119, "ws32x128x4c4p_k32_s4"),       # 10.6, 8.9
    (19136, 216, 384, 64, 0.020, "ws64x64x4c4p_k32_s3"),        # 9.5, 8.2
    (12288, 114, 2352, 128, 0.311, "ws128x32x4c4p_k32_s4"),     # 42.3, 35.9
])
def test_choice_with_and_without_c(torch_gpu, M, K, N, V, d, slow):
    torch = torch_gpu
    w = P.make_weight(M, K, V, d, True, 13, integer=True)
    B, C = P.make_dense(K, N, 5, integer=True), P.make_dense(M, N, 5, integer=True, stream=3)
    mat = P.upload_weight(w)
    b, c, out = (torch.empty((r, N), dtype=torch.float16, device="cuda") for r in (K, M, M))
    added = S.SpmmBlockwiseOp().initialize(mat, N, b.data_ptr(), out.data_ptr(), c.data_ptr()).variant
    assert S.spmm_variants(V)[added] != slow
    for x, beta in ((None, 0.0), (C, 1.0)):
        ref = O.float_to_half(P.spmm_oracle(w, B, x, 1.0, beta))
        got = run_spmm(torch, w, B, Cmat=x, variant=-1)
        np.testing.assert_array_equal(got.view(np.uint16), ref.view(np.uint16))


@pytest.mark.parametrize("M,K,N,V,d,slow", [
    # large results under narrow tiles, more than the Infinity Cache holds
    (12416, 69, 63096, 128, 0.053, "ws128x32x4c4p_k32_s4"),     # 794 us, fastest 553
    (1664, 509, 116576, 128, 0.094, "ws128x32x4c4p_k32_s4"),    # 163, 119
    (5952, 744, 64552, 64, 0.095, "ws64x64x4c4p_k32_s3"),       # 340, 299
    (36064, 286, 34376, 32, 0.044, "ws32x64x4c4p_k32_s3"),      # 1018, 760
    # long panels, a few compute units with two of them
    (5472, 3207, 368, 32, 0.374, "ws32x32x4c4p_k32_s6"),        # 19.2, 15.7
    (1632, 3869, 744, 32, 0.443, "ws32x32x4c4p_k32_s6"),        # 17.4, 14.3
    # few tiles: the split form's reduction costs more than it saves
    (2784, 4288, 8, 32, 0.051, "split32x32"),                   # 4.7, 4.0
])
def test_not_the_slow_variant(torch_gpu, M, K, N, V, d, slow):
    mat = P.upload_weight(P.make_weight(M, K, V, d, True, 13, integer=True))
    t = torch_gpu.zeros(64, dtype=torch_gpu.float16, device="cuda")  # never touched: nothing is launched
    taken = S.SpmmBlockwiseOp().initialize(mat, N, t.data_ptr(), t.data_ptr()).variant
    assert S.spmm_variants(V)[taken] != slow
