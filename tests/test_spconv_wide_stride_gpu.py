"""Strides far wider than the map.  The plane forms hold stride^2 planes and refuse what does not fit, also where that number
leaves the integers it is computed in (initialisation only: nothing is launched on what it accepts)."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S
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
