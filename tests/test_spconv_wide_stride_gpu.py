"""Strides far wider than the map.  The plane forms hold stride^2 planes and refuse what does not fit, also where that number
leaves the integers it is computed in (initialisation only: nothing is launched on what it accepts).  The batch-innermost form
over the input itself has no planes and takes every stride, as long as the rows of the input it computes are integers."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S
from oracle import oracle as O
from shflbw_sparse_nn_amd import capi
import workloads as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", [0, 2, 3])
@pytest.mark.parametrize("stride", [5793, 46341, 1 << 16, 1 << 30, (1 << 31) - 1])
def test_plane_forms_refuse_too_many_planes(torch_gpu, form, stride):
    C, V = 16, 32
    f = P.upload_weight(P.make_weight(64, 9 * C, V, 0.3, True, 3, integer=True), 3, 3, C, cls=S.BlockwiseSpFilter)
    t = torch_gpu.zeros(8 * 8 * 8 * 64, dtype=torch_gpu.float16, device="cuda")
    with pytest.raises(capi.ShflbwError) as e:
        S.SpconvBlockwiseOp(form).initialize(f, 8, 8, 8, stride, t.data_ptr(), t.data_ptr())
    assert e.value.status == capi.ERR_UNSUPPORTED


@pytest.mark.parametrize("H,W", [(7, 9), (8, 5), (1, 12)])
@pytest.mark.parametrize("stride", [8, 100, 1 << 23, 1 << 29, 1 << 30, (1 << 31) - 1])
def test_batch_innermost(torch_gpu, H, W, stride):
    """Only the first position of a row and of a column reads the map (multiplied out in 32 bits, the fifth row at stride 2^30
    would be row 0 again)."""
    torch = torch_gpu
    Bn, C, F = 8, 16, 64
    w = P.make_weight(F, 9 * C, 32, 0.3, True, 3, integer=True)
    x = np.random.default_rng(9).integers(1, 5, size=(C, H, W, Bn)).astype(np.float16)
    f = P.upload_weight(w, 3, 3, C, cls=S.BlockwiseSpFilter)
    dX, dY = P.to_dev(torch, x), torch.full((F, H, W, Bn), float("nan"), dtype=torch.float16, device="cuda")
    op = S.SpconvBlockwiseOp()
    op.initialize(f, Bn, H, W, stride, dX.data_ptr(), dY.data_ptr(), batch_innermost=True)
    op(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    # the oracle at a stride past the map that its integers hold
    ref = O.float_to_half(P.conv_oracle_batch_first(w, 3, 3, C, x, min(stride, 1000)))
    np.testing.assert_array_equal(dY.cpu().numpy().view(np.uint16), ref.view(np.uint16))


def test_batch_innermost_refuses_positions_beyond_an_int(torch_gpu):
    """2^20 rows at a stride of 2^12: input rows up to 2^32.  Neither the input nor planes of it can be gathered from."""
    f = P.upload_weight(P.make_weight(16, 9, 16, 1.0, False, 3, integer=True), 3, 3, 1, cls=S.BlockwiseSpFilter)
    t = torch_gpu.zeros(64, dtype=torch_gpu.float16, device="cuda")  # never touched: the initialisation fails
    with pytest.raises(capi.ShflbwError) as e:
        S.SpconvBlockwiseOp().initialize(f, 8, 1 << 20, 1, 1 << 12, t.data_ptr(), t.data_ptr() + (1 << 32), batch_innermost=True)
    assert e.value.status == capi.ERR_UNSUPPORTED
