"""The batch-innermost convolution (C-H-W-B in, F-H-W-B out): the launch that gathers from the input itself, in the cuts that the
library takes, at the edges of its rule (31 taps, overlapping tensors), bit for bit on integer data against the oracle.  Its
kernels, each by name: tests/cpp/test_chwb_cuts.cc."""
import numpy as np
import pytest

import workloads as P
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Bn,H,W,C,F,R,S,stride,V,d,planes", [
    (8, 1, 1, 1, 16, 3, 3, 1, 16, 1.0, False),       # one position: every outer tap reads zeros
    (8, 9, 40, 3, 32, 1, 31, 1, 32, 0.5, False),     # as many taps as a lane keeps bits for
    (8, 9, 17, 3, 32, 4, 8, 1, 32, 0.5, True),       # one more: planes
    (16, 11, 6, 5, 64, 7, 7, 2, 64, 0.3, True),
    (40, 13, 7, 12, 128, 5, 5, 2, 128, 0.2, False),  # tiles whose pieces belong to several positions
    (128, 14, 14, 16, 256, 3, 3, 1, 64, 0.1, False),
    (64, 14, 14, 9, 256, 3, 3, 3, 32, 0.3, False),   # tiles of 256 columns
    (24, 30, 30, 7, 640, 2, 4, 1, 64, 0.2, False),   # even extents, a ragged last tile
    (104, 15, 15, 4, 48, 1, 1, 2, 16, 0.9, False),
    (8, 5, 6, 70, 64, 3, 1, 2, 32, 0.0, False),      # panels that keep next to nothing
])
def test_chwb_exact(torch_gpu, Bn, H, W, C, F, R, S, stride, V, d, planes):
    import shflbw_sparse_nn_amd as Sx
    torch = torch_gpu
    w = P.make_weight(F, R * S * C, V, d, True, 2021, integer=True)
    x = np.random.default_rng(9).integers(-4, 5, size=(C, H, W, Bn)).astype(np.float16)
    ref = O.float_to_half(P.conv_oracle_batch_first(w, R, S, C, x, stride))
    f = P.upload_weight(w, R, S, C, cls=Sx.BlockwiseSpFilter)
    dX = P.to_dev(torch, x)
    dY = torch.full((F, H, W, Bn), float("nan"), dtype=torch.float16, device="cuda")
    op = Sx.SpconvBlockwiseOp()
    st = op.initialize(f, Bn, H, W, stride, dX.data_ptr(), dY.data_ptr(), batch_innermost=True)
    assert bool(st.planes) == planes
    op(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(dY.cpu().numpy().view(np.uint16), ref.view(np.uint16))


def test_chwb_in_place(torch_gpu):
    """An output that lies over the input takes the form that copies the input first."""
    import shflbw_sparse_nn_amd as Sx
    torch = torch_gpu
    Bn, H, W, C, F = 16, 9, 9, 64, 64
    w = P.make_weight(F, 9 * C, 32, 0.2, True, 5, integer=True)
    x = np.random.default_rng(3).integers(-4, 5, size=(C, H, W, Bn)).astype(np.float16)
    ref = O.float_to_half(P.conv_oracle_batch_first(w, 3, 3, C, x, 1))
    f = P.upload_weight(w, 3, 3, C, cls=Sx.BlockwiseSpFilter)
    t = P.to_dev(torch, x)
    op = Sx.SpconvBlockwiseOp()
    st = op.initialize(f, Bn, H, W, 1, t.data_ptr(), t.data_ptr(), batch_innermost=True)
    assert st.planes
    op(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(t.cpu().numpy().reshape(F, H, W, Bn).view(np.uint16), ref.view(np.uint16))


def test_chwb_non_finite(torch_gpu):
    """Infinities and NaN in the input reach the outputs whose kept taps read them, and no others."""
    import shflbw_sparse_nn_amd as Sx
    torch = torch_gpu
    Bn, H, W, C, F, R, S = 8, 6, 7, 10, 64, 3, 3
    w = P.make_weight(F, R * S * C, 32, 0.3, True, 5, integer=True)
    x = np.random.default_rng(3).integers(-4, 5, size=(C, H, W, Bn)).astype(np.float16)
    x[2, 0, 0, 1], x[5, 5, 6, 7], x[9, 3, 3, 0] = np.inf, np.nan, -np.inf
    with np.errstate(invalid="ignore", over="ignore"):
        ref = O.float_to_half(P.conv_oracle_batch_first(w, R, S, C, x, 1))
    f = P.upload_weight(w, R, S, C, cls=Sx.BlockwiseSpFilter)
    dX = P.to_dev(torch, x)
    dY = torch.zeros((F, H, W, Bn), dtype=torch.float16, device="cuda")
    op = Sx.SpconvBlockwiseOp()
    op.initialize(f, Bn, H, W, 1, dX.data_ptr(), dY.data_ptr(), batch_innermost=True)
    op(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = dY.cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    np.testing.assert_array_equal(got[~np.isnan(ref)], ref[~np.isnan(ref)])
