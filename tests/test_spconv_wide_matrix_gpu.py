"""Convolutions whose im2col matrix (R*S*C x output positions, which is never built) would exceed 4 GiB while the input and its planes
do not: every form that gathers by ids takes them, block height 16 too, whose kernels have 32-bit offsets only.  Integer
operands, bit for bit against the oracle."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S
from oracle import oracle as O
import workloads as P

pytestmark = pytest.mark.gpu
CHWB = 4


@pytest.mark.parametrize("form,V", [(CHWB, 16), (2, 16), (3, 16), (0, 16), (0, 32)])
def test_im2col_matrix_beyond_4_gib(torch_gpu, form, V):
    torch = torch_gpu
    Bn, H, W, C, F, R = 128, 40, 40, 424, 32, 5
    assert R * R * C * H * W * Bn * 2 > 2 ** 32
    w = P.make_weight(F, R * R * C, V, 0.003, True, 7, integer=True)
    x = np.random.default_rng(3).integers(-4, 5, size=(C, H, W, Bn) if form == CHWB else (Bn, H, W, C), dtype=np.int8).astype(np.float16)
    f = P.upload_weight(w, R, R, C, cls=S.BlockwiseSpFilter)
    dX = P.to_dev(torch, x)
    dY = torch.full((F, H, W, Bn) if form == CHWB else (Bn, H, W, F), float("nan"), dtype=torch.float16, device="cuda")
    op = S.SpconvBlockwiseOp(-1 if form == CHWB else form)
    st = op.initialize(f, Bn, H, W, 1, dX.data_ptr(), dY.data_ptr(), batch_innermost=form == CHWB)
    assert st.variant == form
    op(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    op.check()
    ref = O.float_to_half(P.conv_oracle_batch_first(w, R, R, C, x, 1) if form == CHWB else P.conv_oracle(w, R, R, C, x, 1))
    np.testing.assert_array_equal(dY.cpu().numpy().view(np.uint16), ref.view(np.uint16))
