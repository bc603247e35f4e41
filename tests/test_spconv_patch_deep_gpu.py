"""The patch form's kernels with more batches in flight, which waves with many batches run: every row unit that has one, as many
batches as the rule asks for and fewer, parts of the kept columns and several row units a wave, panels that keep nothing."""
import numpy as np
import pytest

import shflbw_sparse_nn_amd as S
from oracle import oracle as O
import workloads as P
from workloads import run_spconv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Bn,H,W,C,F,R,stride,V,d,permute", [
    (2, 20, 21, 136, 96, 3, 1, 32, 0.25, True),
    (3, 14, 30, 224, 320, 3, 2, 32, 0.22, False),
    (8, 11, 10, 72, 256, 1, 1, 32, 1.0, True),
    (4, 22, 20, 24, 160, 3, 1, 16, 0.445, True),
    (3, 13, 26, 48, 304, 3, 2, 16, 0.398, True),
    (2, 9, 9, 512, 16, 1, 1, 16, 0.9, True),
])
def test_deep_ring(torch_gpu, Bn, H, W, C, F, R, stride, V, d, permute):
    w = P.make_weight(F, R * R * C, V, d, permute, 2021, integer=True)
    x = np.random.default_rng(5).integers(-4, 5, size=(Bn, H, W, C)).astype(np.float16)

    def check(w):
        got = run_spconv(torch_gpu, w, R, R, C, x, stride, 5)
        ref = O.float_to_half(P.conv_oracle(w, R, R, C, x, stride))
        np.testing.assert_array_equal(got.view(np.uint16), ref.view(np.uint16))

    check(w)
    counts = np.diff(w["indptr"])
    counts[1::3] = 0  # ... and uneven panels, some without a kept column
    counts[::4] = np.maximum(counts[::4] // 3, 1)
    sel = np.concatenate([np.arange(b, b + n) for b, n in zip(w["indptr"], counts)]).astype(np.int64)
    check(dict(w, nnzb=int(counts.sum()), indptr=np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), indices=w["indices"][sel],
               values=w["values"].reshape(-1, V)[sel].reshape(-1)))
