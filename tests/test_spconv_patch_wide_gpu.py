"""The patch form's wide cuts: a permuted filter of more than 512 rows whose results leave from one workgroup, each wave computing
several row units one after the other that go to LDS as they are finished.  Every block height, the fewest and the most units of a
wave, a last wave with fewer of them or none, pixels that do not fill the last tile, and panels that keep nothing (also all of a
wave's, the first and the last).  Strides, filters of one row, strides wider than the filter.  Integer operands, bit for bit against the CPU oracle."""
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle as O
import workloads as P
from workloads import run_spconv

pytestmark = pytest.mark.gpu
PLAN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin", "test_patch_plan")
WIDE = 2  # last figure of a cut


def _cut(w, R, C, x, stride, Sx=None):
    """(32-column blocks, row units of a wave, workgroups per column tile, kernel) of the cut that the planner picks"""
    args = [w["brow"], w["nrow"], C, R, Sx or R, w["nnzb"], 1, *x.shape[:3], stride]
    v = list(map(int, subprocess.check_output([PLAN, "cut"] + [str(int(a)) for a in args], text=True).split()))
    return v[1], v[3], v[5], v[6]


@pytest.mark.parametrize("blocks,units,Bn,H,W,C,F,R,stride,V,d", [
    (1, 5, 20, 19, 13, 72, 576, 3, 1, 16, 0.1),
    (1, 7, 20, 19, 15, 224, 800, 3, 1, 16, 0.1),
    (1, 8, 20, 19, 13, 120, 1008, 1, 1, 16, 0.1),
    (1, 15, 20, 17, 13, 120, 1920, 1, 1, 16, 0.1),
    (2, 5, 56, 14, 13, 72, 528, 1, 1, 16, 0.05),
    (2, 8, 40, 17, 13, 32, 1008, 1, 1, 16, 0.05),
    (2, 3, 40, 14, 15, 16, 576, 1, 1, 32, 0.1),
    (2, 4, 64, 17, 8, 24, 1024, 3, 1, 32, 0.1),
    (2, 2, 64, 19, 13, 16, 1024, 3, 1, 64, 0.1),
    (2, 2, 40, 17, 13, 16, 1024, 3, 1, 128, 0.1),
    (1, 3, 20, 17, 13, 24, 672, 1, 1, 32, 0.2),
    (1, 4, 20, 14, 15, 152, 1024, 3, 1, 32, 0.05),
    (1, 7, 20, 19, 15, 104, 1600, 3, 1, 32, 0.2),
    (1, 8, 20, 17, 15, 208, 1824, 1, 1, 32, 0.1),
    (1, 2, 20, 19, 13, 120, 1024, 1, 1, 64, 0.1),
    (1, 3, 20, 17, 13, 144, 1088, 1, 1, 64, 0.1),
    (1, 4, 20, 19, 15, 88, 1664, 1, 1, 64, 0.2),
    (1, 2, 20, 19, 15, 184, 1024, 1, 1, 128, 0.05),
    (1, 3, 20, 19, 15, 16, 1152, 3, 1, 128, 0.2),
    (1, 4, 20, 14, 13, 184, 1664, 1, 1, 128, 0.1),
    (1, 3, 30, 28, 28, 16, 1344, 1, 1, 64, 0.135),  # 63 MB of output: streaming stores
])
def test_all_filters_in_one_workgroup(torch_gpu, blocks, units, Bn, H, W, C, F, R, stride, V, d):
    w = P.make_weight(F, R * R * C, V, d, True, 2021, integer=True)
    x = np.random.default_rng(5).integers(-4, 5, size=(Bn, H, W, C)).astype(np.float16)
    assert _cut(w, R, C, x, stride) == (blocks, units, 1, WIDE)
    X, counts = F // V, np.diff(w["indptr"])
    for gone in ((), range(0, X, 3), range(X // 3, X), range(X - X // 3)):
        kept = counts.copy()
        kept[list(gone)] = 0
        sel = np.concatenate([np.arange(b, b + n) for b, n in zip(w["indptr"], kept)]).astype(np.int64)
        w2 = dict(w, nnzb=int(kept.sum()), indptr=np.concatenate([[0], np.cumsum(kept)]).astype(np.int32),
                  indices=w["indices"][sel], values=w["values"].reshape(-1, V)[sel].reshape(-1))
        if gone == () or _cut(w2, R, C, x, stride)[3] == WIDE:
            got = run_spconv(torch_gpu, w2, R, R, C, x, stride, 5)
            ref = O.float_to_half(P.conv_oracle(w2, R, R, C, x, stride))
            np.testing.assert_array_equal(got.view(np.uint16), ref.view(np.uint16))


@pytest.mark.parametrize("blocks,units,Bn,H,W,C,F,R,Sx,stride,V,d", [
    (1, 5, 12, 25, 28, 80, 640, 3, 3, 2, 16, 0.05),
    (2, 5, 24, 25, 20, 160, 640, 1, 7, 1, 16, 0.1),
    (1, 5, 33, 26, 20, 8, 528, 1, 7, 2, 16, 0.2),
    (2, 5, 40, 26, 28, 72, 576, 5, 5, 2, 16, 0.05),
    (1, 4, 33, 26, 30, 144, 832, 3, 3, 2, 32, 0.2),
    (2, 3, 40, 25, 26, 64, 640, 1, 7, 2, 32, 0.1),
    (1, 4, 40, 23, 24, 80, 800, 1, 1, 2, 32, 0.05),
    (1, 3, 20, 29, 14, 40, 1344, 1, 7, 1, 64, 0.1),
    (1, 4, 12, 29, 29, 112, 1600, 3, 3, 2, 64, 0.05),
    (2, 2, 40, 26, 28, 32, 1024, 1, 1, 2, 64, 0.2),
    (1, 2, 40, 24, 24, 120, 640, 3, 3, 3, 128, 0.1),
    (2, 2, 40, 29, 29, 56, 1024, 1, 7, 2, 128, 0.05),
])
def test_strides_and_shapes_of_filters(torch_gpu, blocks, units, Bn, H, W, C, F, R, Sx, stride, V, d):
    w = P.make_weight(F, R * Sx * C, V, d, True, 2021, integer=True)
    x = np.random.default_rng(5).integers(-4, 5, size=(Bn, H, W, C)).astype(np.float16)
    assert _cut(w, R, C, x, stride, Sx) == (blocks, units, 1, WIDE)
    got = run_spconv(torch_gpu, w, R, Sx, C, x, stride, 5)
    ref = O.float_to_half(P.conv_oracle(w, R, Sx, C, x, stride))
    np.testing.assert_array_equal(got.view(np.uint16), ref.view(np.uint16))
