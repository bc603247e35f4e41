"""The patch form's kernels with more batches in flight, which waves with many batches run: each of them (the cut that the planner
picks is checked, its last figure says which ring), one row unit a wave, several, and parts of the kept columns; then the same
layers with panels that keep nothing, one batch, and as many as fill the ring, one less and one more.  And cuts with as few batches
a wave as stay with the short ring."""
import os
import subprocess

import numpy as np
import pytest

from oracle import oracle as O
import workloads as P
from workloads import run_spconv

pytestmark = pytest.mark.gpu
PLAN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin", "test_patch_plan")
RING = {(16, 1): 6, (32, 1): 4, (32, 2): 6}  # batches in flight, by rows of a row unit and 32-column blocks


def _cut(w, R, C, x, stride):
    """(rows of a row unit, 32-column blocks, waves, row units of a wave, parts of the kept columns, deep ring)"""
    args = [w["brow"], w["nrow"], C, R, R, w["nnzb"], int(w["row_permute_ids"] is not None), *x.shape[:3], stride]
    v = list(map(int, subprocess.check_output([PLAN, "cut"] + [str(int(a)) for a in args], text=True).split()))
    return tuple(v[:5] + v[6:])


def _uneven(w, ring, turn):
    """The same number of kept columns, but up to half of the panels keep 0, 1, ring - 1, ring, ring + 1, ... batches of 32."""
    X, K = w["nrow"] // w["brow"], w["ncol"]
    rng = np.random.default_rng(turn)
    edges = np.roll([0, 1, ring - 1, ring, ring + 1, 2 * ring, 2 * ring + 1], -turn)[:X // 2]
    counts = np.zeros(X, np.int64)
    counts[:len(edges)] = np.maximum(32 * edges - rng.integers(0, 32, len(edges)), 0)
    rest, others = w["nnzb"] - counts.sum(), X - len(edges)
    counts[len(edges):] = rest // others + (np.arange(others) < rest % others)
    assert (counts <= K).all()
    counts = rng.permutation(counts)
    indices = np.concatenate([np.sort(rng.choice(K, n, replace=False)) for n in counts])
    return dict(w, indptr=np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), indices=indices.astype(np.int32))


@pytest.mark.parametrize("cut,Bn,H,W,C,F,R,stride,V,d,permute", [
    ((16, 1, 4, 1, 1, 1), 7, 4, 22, 216, 48, 3, 1, 16, 0.211, True),   # 13 batches a wave, the fewest
    ((16, 1, 4, 1, 1, 1), 7, 9, 20, 112, 64, 5, 2, 16, 0.149, True),
    ((16, 1, 4, 1, 2, 1), 1, 12, 7, 48, 48, 5, 2, 16, 0.66, True),
    ((16, 1, 4, 1, 4, 1), 1, 14, 6, 400, 16, 3, 2, 16, 0.804, True),
    ((16, 1, 4, 2, 1, 1), 12, 29, 9, 192, 96, 3, 2, 16, 0.118, True),
    ((16, 1, 4, 4, 1, 1), 9, 15, 16, 136, 224, 3, 1, 16, 0.108, True),
    ((32, 1, 4, 1, 1, 1), 9, 8, 12, 72, 96, 5, 1, 32, 0.16, True),
    ((32, 1, 4, 1, 2, 1), 1, 5, 6, 232, 64, 3, 1, 32, 0.248, True),    # 9
    ((32, 1, 4, 1, 4, 1), 1, 5, 14, 136, 32, 3, 2, 32, 0.942, True),
    ((32, 1, 4, 2, 1, 1), 8, 26, 7, 184, 160, 3, 1, 32, 0.109, True),
    ((32, 2, 4, 1, 1, 1), 8, 19, 24, 136, 96, 3, 1, 32, 0.262, True),
    ((32, 2, 4, 1, 2, 1), 9, 17, 28, 120, 96, 3, 1, 32, 0.613, True),
    ((32, 2, 4, 1, 4, 1), 1, 7, 14, 464, 32, 3, 2, 32, 0.973, True),
    ((32, 2, 4, 2, 1, 1), 12, 24, 29, 112, 256, 3, 1, 32, 0.129, True),
    ((32, 1, 4, 1, 4, 0), 2, 20, 21, 136, 96, 3, 1, 32, 0.25, True),
    ((32, 1, 4, 1, 4, 0), 3, 14, 30, 224, 320, 3, 2, 32, 0.22, False),
    ((32, 1, 4, 1, 4, 0), 8, 11, 10, 72, 256, 1, 1, 32, 1.0, True),
    ((16, 1, 4, 1, 4, 0), 4, 22, 20, 24, 160, 3, 1, 16, 0.445, True),
    ((16, 1, 4, 1, 4, 0), 3, 13, 26, 48, 304, 3, 2, 16, 0.398, True),
    ((16, 1, 4, 1, 4, 0), 2, 9, 9, 512, 16, 1, 1, 16, 0.9, True),
])
def test_deep_ring(torch_gpu, cut, Bn, H, W, C, F, R, stride, V, d, permute):
    w = P.make_weight(F, R * R * C, V, d, permute, 2021, integer=True)
    x = np.random.default_rng(5).integers(-4, 5, size=(Bn, H, W, C)).astype(np.float16)
    for weight in [w] + [_uneven(w, RING[cut[:2]], turn) for turn in (0, 2, 4) if cut[5] and F > V]:
        assert _cut(weight, R, C, x, stride) == cut
        got = run_spconv(torch_gpu, weight, R, R, C, x, stride, 5)
        ref = O.float_to_half(P.conv_oracle(weight, R, R, C, x, stride))
        np.testing.assert_array_equal(got.view(np.uint16), ref.view(np.uint16))
