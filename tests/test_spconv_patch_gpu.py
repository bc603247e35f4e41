"""GPU parity of the patch form of the convolution (one launch, the input patch of a workgroup in LDS) against the CPU
oracle: integer operands, bit for bit.  The shapes sit where the form can go wrong: edges of the pixel blocks and of the
four-unit tiles, channel counts that leave part of a 64-channel group, strides wider than the filter, every block
height, one and several workgroups per column tile with and without a permutation, kept columns split over waves; and, by
the cut that the planner picks, every kernel of the form, several row units a wave and every number of parts."""
import os
import subprocess

import numpy as np
import pytest

import shflbw_sparse_nn_amd as S
from oracle import oracle as O
import workloads as P
from workloads import run_spconv

pytestmark = pytest.mark.gpu
PATCH = 5


def _check(torch, w, x, R, Sx, C, stride):
    got = run_spconv(torch, w, R, Sx, C, x, stride, PATCH)
    with np.errstate(invalid="ignore", over="ignore"):
        ref = O.float_to_half(P.conv_oracle(w, R, Sx, C, x, stride))
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got[~nan].view(np.uint16), ref[~nan].view(np.uint16))


@pytest.mark.parametrize("Bn,H,W,C,F,R,Sx,stride,V,d,permute", [
    (1, 1, 1, 8, 16, 1, 1, 1, 16, 1.0, True),          # one pixel, one panel
    (1, 5, 5, 8, 32, 3, 3, 1, 32, 0.5, True),          # fewer blocks than a tile has units
    (3, 9, 9, 8, 128, 1, 1, 1, 128, 0.6, False),       # 1 x 1: one long row of pixels over all images
    (2, 8, 8, 24, 64, 5, 3, 1, 32, 0.2, True),         # three groups of eight channels
    (2, 9, 7, 16, 48, 3, 3, 1, 16, 0.4, True),
    (1, 11, 9, 16, 64, 3, 3, 3, 64, 0.5, True),
    (2, 6, 20, 8, 32, 1, 7, 1, 32, 0.4, True),
    (8, 9, 8, 16, 64, 4, 2, 2, 32, 0.3, True),         # even filter extents
    (5, 9, 9, 40, 704, 1, 1, 2, 64, 0.25, True),       # stride wider than the filter, eleven panels
    (5, 13, 3, 136, 64, 2, 2, 3, 64, 0.25, True),
    (3, 9, 9, 40, 2048, 3, 3, 1, 16, 0.25, True),      # filters of several workgroups interleaved in a pixel
    (3, 9, 9, 40, 1536, 3, 3, 1, 128, 0.25, True),
    (3, 9, 9, 40, 1088, 3, 3, 1, 32, 0.25, False),     # ... consecutive
    (1, 7, 7, 512, 64, 3, 3, 1, 64, 0.1, True),        # one panel: its kept columns over all waves of a workgroup
    (2, 30, 31, 32, 96, 3, 3, 1, 32, 0.02, True),      # panels with almost no kept column
    (24, 28, 28, 32, 64, 3, 3, 1, 64, 0.2, True),      # several workgroups of a compute unit at a time
])
def test_exact_shapes(torch_gpu, Bn, H, W, C, F, R, Sx, stride, V, d, permute):
    w = P.make_weight(F, R * Sx * C, V, d, permute, 2021, integer=True)
    x = np.random.default_rng(5).integers(-4, 5, size=(Bn, H, W, C)).astype(np.float16)
    _check(torch_gpu, w, x, R, Sx, C, stride)


def _cut(w, R, Sx, C, x, stride):
    """(rows of a row unit, 32-column blocks, waves, row units of a wave, parts of the kept columns) the planner picks."""
    exe = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "bin", "test_patch_plan")
    args = [w["brow"], w["nrow"], C, R, Sx, w["nnzb"], int(w["row_permute_ids"] is not None), *x.shape[:3], stride]
    return tuple(map(int, subprocess.check_output([exe, "cut"] + [str(int(a)) for a in args], text=True).split()))[:5]


@pytest.mark.parametrize("cut,Bn,H,W,C,F,R,stride,V,d,permute", [
    ((16, 1, 4, 2, 1), 29, 10, 17, 160, 96, 3, 2, 16, 0.05, True),
    ((16, 1, 4, 4, 1), 18, 30, 25, 80, 144, 3, 1, 16, 0.1, True),
    ((16, 2, 4, 2, 1), 15, 22, 25, 80, 80, 3, 1, 16, 0.1, True),
    ((16, 2, 4, 4, 1), 27, 20, 25, 56, 176, 5, 1, 16, 0.05, True),
    ((16, 1, 8, 1, 1), 13, 8, 26, 264, 128, 3, 2, 16, 0.05, True),
    ((16, 1, 8, 1, 4), 11, 15, 11, 232, 32, 5, 2, 16, 0.05, True),
    ((16, 1, 8, 2, 1), 24, 19, 17, 168, 144, 3, 2, 16, 0.05, True),
    ((16, 1, 8, 4, 1), 18, 28, 22, 160, 320, 3, 2, 16, 0.05, True),
    ((16, 2, 8, 1, 1), 37, 28, 30, 168, 80, 3, 2, 16, 0.05, True),
    ((16, 2, 8, 1, 8), 36, 15, 15, 136, 16, 5, 1, 16, 0.05, True),
    ((16, 2, 8, 2, 1), 22, 28, 13, 160, 144, 3, 1, 16, 0.05, True),
    ((16, 2, 8, 4, 1), 35, 19, 13, 160, 272, 3, 1, 16, 0.05, True),
    ((32, 1, 4, 2, 1), 29, 9, 15, 192, 160, 3, 2, 32, 0.05, True),
    ((32, 2, 4, 2, 1), 14, 21, 25, 56, 160, 5, 1, 32, 0.05, True),
    ((32, 1, 8, 1, 2), 28, 20, 10, 232, 288, 3, 2, 32, 0.05, True),
    ((32, 1, 8, 1, 8), 1, 4, 6, 280, 32, 5, 2, 32, 0.2, True),
    ((32, 1, 8, 2, 1), 20, 26, 11, 208, 288, 3, 2, 32, 0.05, True),
    ((32, 2, 8, 1, 1), 25, 11, 28, 160, 160, 3, 1, 32, 0.05, False),
    ((32, 2, 8, 1, 4), 26, 10, 5, 272, 544, 3, 1, 32, 0.05, True),
    ((32, 2, 8, 2, 1), 33, 9, 25, 40, 288, 3, 1, 32, 0.2, True),
    ((64, 1, 8, 1, 1), 23, 12, 20, 208, 320, 3, 2, 64, 0.05, True),
    ((64, 1, 8, 1, 4), 27, 15, 25, 264, 128, 3, 2, 64, 0.05, True),
    ((64, 2, 8, 1, 1), 19, 19, 21, 160, 320, 3, 1, 64, 0.05, True),
    ((64, 2, 8, 1, 8), 40, 7, 28, 208, 64, 5, 1, 64, 0.05, True),
    ((64, 2, 8, 1, 4), 40, 28, 31, 272, 128, 3, 2, 128, 0.05, True),
    ((64, 2, 4, 1, 1), 35, 10, 9, 56, 384, 5, 1, 64, 0.05, False),
    ((64, 1, 4, 1, 2), 3, 22, 7, 72, 512, 5, 2, 128, 0.05, False),
])
def test_exact_by_cut(torch_gpu, cut, Bn, H, W, C, F, R, stride, V, d, permute):
    """The 8-wave kernels (deeper ring, more of the patch in flight) and waves with several row units one after the other; the
    third and every fourth panel from there on keep nothing, one other keeps a single column."""
    w = P.make_weight(F, R * R * C, V, d, permute, 2021, integer=True)
    x = np.random.default_rng(5).integers(-4, 5, size=(Bn, H, W, C)).astype(np.float16)
    assert _cut(w, R, R, C, x, stride) == cut
    _check(torch_gpu, w, x, R, R, C, stride)
    X = F // V
    counts = np.diff(w["indptr"])
    counts[2::4] = 0
    counts[X // 2] = min(1, counts[X // 2])
    sel = np.concatenate([np.arange(b, b + n) for b, n in zip(w["indptr"], counts)]).astype(np.int64)
    w2 = dict(w, nnzb=int(counts.sum()), indptr=np.concatenate([[0], np.cumsum(counts)]).astype(np.int32),
              indices=w["indices"][sel], values=w["values"].reshape(-1, V)[sel].reshape(-1))
    if cut[3] > 1:
        assert _cut(w2, R, R, C, x, stride) == cut
    _check(torch_gpu, w2, x, R, R, C, stride)


@pytest.mark.parametrize("V", [16, 32, 64, 128])
def test_empty_panels_and_non_finite_input(torch_gpu, V):
    """Panels without a kept column give zeros; an Inf or NaN in the input reaches the outputs it reaches in the oracle and
    no other (padding slots read a row of zeros)."""
    Bn, H, W, C, R, Sx = 2, 9, 10, 16, 3, 3
    X, K = 6, R * Sx * C
    counts = np.array([0, 33, 0, 5, 64, 0])
    rng = np.random.default_rng(5)
    indptr = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    indices = np.concatenate([np.sort(rng.choice(K, c, replace=False)) for c in counts]).astype(np.int32)
    values = rng.integers(1, 5, size=int(counts.sum()) * V).astype(np.float16)  # no zero: 0 * inf is NaN in the oracle too
    w = dict(nrow=X * V, ncol=K, brow=V, bcol=1, nnzb=int(counts.sum()), indptr=indptr, indices=indices, values=values,
             row_permute_ids=O.row_permutation(X * V, 5))
    x = rng.integers(-4, 5, size=(Bn, H, W, C)).astype(np.float16)
    _check(torch_gpu, w, x, R, Sx, C, 1)
    x[0, 4, 5, 3], x[1, 0, 0, 15], x[1, 8, 9, 0] = np.inf, -np.inf, np.nan
    _check(torch_gpu, w, x, R, Sx, C, 1)


def test_the_library_runs_it_and_it_needs_no_buffers(torch_gpu):
    """shflbw_spconv_init takes the patch form on an ordinary layer and the state says so; states over many tensors share its tables;
    weights of too many channels for the LDS keep the plane form."""
    torch = torch_gpu
    w = P.make_weight(64, 9 * 64, 32, 0.2, True, 3, integer=True)
    f = P.upload_weight(w, 3, 3, 64, cls=S.BlockwiseSpFilter)
    x = torch.zeros((8, 14, 14, 64), dtype=torch.float16, device="cuda")
    ops = []
    for _ in range(3):
        op = S.SpconvBlockwiseOp()
        y = torch.full((8, 14, 14, 64), float("nan"), dtype=torch.float16, device="cuda")
        st = op.initialize(f, 8, 14, 14, 1, x.data_ptr(), y.data_ptr())
        assert st.patch and st.variant == PATCH and S.spconv_variant_name(st.variant) == "patch"
        op(torch.cuda.current_stream().cuda_stream)
        ops.append((op, y))
    torch.cuda.synchronize()
    assert len({op._state.patch for op, _ in ops}) == 1 and all((y == 0).all() for _, y in ops)
    wide = P.make_weight(64, 25 * 1024, 64, 0.01, True, 3, integer=True)
    fw = P.upload_weight(wide, 5, 5, 1024, cls=S.BlockwiseSpFilter)
    xw = torch.zeros((1, 8, 8, 1024), dtype=torch.float16, device="cuda")
    op = S.SpconvBlockwiseOp()
    st = op.initialize(fw, 1, 8, 8, 1, xw.data_ptr(), ops[0][1].data_ptr())
    assert not st.patch and st.variant == 0


@pytest.mark.parametrize("Bn,H,C,F,V,stride", [(1, 5, 512, 64, 64, 2), (4, 8, 512, 128, 128, 2)])
def test_variant_5_runs_where_the_library_would_not_choose_it(torch_gpu, Bn, H, C, F, V, stride):
    """A layer whose patch fits the LDS but whose plane forms are estimated faster: the library takes a plane form, an explicit
    request runs the patch form, and neither changes what the other gets."""
    torch = torch_gpu
    w = P.make_weight(F, 25 * C, V, 0.4, True, 3, integer=True)
    x = np.random.default_rng(5).integers(-4, 5, size=(Bn, H, H, C)).astype(np.float16)
    ref = O.float_to_half(P.conv_oracle(w, 5, 5, C, x, stride))
    f = P.upload_weight(w, 5, 5, C, cls=S.BlockwiseSpFilter)
    dX = P.to_dev(torch, x)
    for variant in (-1, PATCH, -1, PATCH):
        dY = torch.full(ref.shape, float("nan"), dtype=torch.float16, device="cuda")
        op = S.SpconvBlockwiseOp(variant)
        st = op.initialize(f, Bn, H, H, stride, dX.data_ptr(), dY.data_ptr())
        assert (st.variant == PATCH) == (variant == PATCH) and st.variant in (0, PATCH)
        op(torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(dY.cpu().numpy().view(np.uint16), ref.view(np.uint16))


def test_variant_5_is_refused_where_no_patch_fits(torch_gpu):
    w = P.make_weight(64, 25 * 1024, 64, 0.01, True, 3, integer=True)
    with pytest.raises(S.capi.ShflbwError) as e:
        run_spconv(torch_gpu, w, 5, 5, 1024, np.zeros((1, 8, 8, 1024), dtype=np.float16), 1, PATCH)
    assert e.value.status == S.capi.ERR_UNSUPPORTED and "LDS" in str(e.value)


@pytest.mark.parametrize("Bn,H,C,F,V,d,stride", [(1, 28, 128, 128, 32, 0.25, 1), (16, 14, 512, 2048, 64, 0.1, 1),
                                                 (32, 28, 256, 512, 32, 0.3, 2), (16, 28, 64, 256, 16, 0.25, 1)])
def test_first_initialisation_of_a_filter_costs_no_more_than_the_plane_form(torch_gpu, Bn, H, C, F, V, d, stride):
    """A program that meets a new filter pays for its tables in the call: planning, ordering and packing the patch form's
    image stay below what the plane form's first initialisation takes (medians over new filters, in turn, which stay alive as
    those of a network do; half as much again is allowed for noise of the host)."""
    import time
    torch = torch_gpu
    w = P.make_weight(F, 9 * C, V, d, True, 3, integer=True)
    dX = torch.zeros((Bn, H, H, C), dtype=torch.float16, device="cuda")
    dY = torch.zeros((Bn, H, H, F), dtype=torch.float16, device="cuda")
    took, alive = {PATCH: [], 0: []}, []
    for _ in range(31):
        for variant in took:
            f = P.upload_weight(w, 3, 3, C, cls=S.BlockwiseSpFilter)
            op = S.SpconvBlockwiseOp(variant)
            alive.append(op)
            torch.cuda.synchronize()
            t = time.perf_counter()
            op.initialize(f, Bn, H, H, stride, dX.data_ptr(), dY.data_ptr())
            took[variant].append(time.perf_counter() - t)
    patch, planes = (np.median(took[v][10:]) * 1e6 for v in (PATCH, 0))
    print("first initialisation: patch form %.0f us, plane form %.0f us" % (patch, planes), flush=True)
    assert patch < 1.5 * planes


def test_a_filter_serves_many_geometries_from_a_bounded_number_of_images(torch_gpu):
    """A serving loop over many batches and resolutions: geometries whose patches have one shape share an image of the filter,
    a filter holds at most SHFLBW_CONV_PATCH_IMAGES (16), and a geometry met after that runs on one of those.  What is held
    does not grow on a second round, and a state made first is still good at the end."""
    import ctypes
    torch = torch_gpu
    C, F, V = 24, 64, 16
    w = P.make_weight(F, 9 * C, V, 0.3, True, 3, integer=True)
    f = P.upload_weight(w, 3, 3, C, cls=S.BlockwiseSpFilter)
    stream = torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(5)

    def held():
        b, n = ctypes.c_size_t(0), ctypes.c_int(0)
        S.capi.check(S.capi.load().shflbw_weight_scratch_bytes(f._h, ctypes.byref(b), ctypes.byref(n)))
        return b.value, n.value

    first, images, sizes = None, set(), []
    for rnd in range(2):
        for stride, H in ((1, 4), (2, 9), (1, 5), (2, 14), (1, 7), (2, 25), (1, 10), (1, 14), (2, 30), (1, 20), (1, 28), (1, 33)):
            for Bn in (1, 2, 3, 5, 8, 13, 24):
                x = rng.integers(-4, 5, size=(Bn, H, H + 1, C)).astype(np.float16)
                ref = O.float_to_half(P.conv_oracle(w, 3, 3, C, x, stride))
                dX, dY = P.to_dev(torch, x), torch.full(ref.shape, float("nan"), dtype=torch.float16, device="cuda")
                op = S.SpconvBlockwiseOp()
                st = op.initialize(f, Bn, H, H + 1, stride, dX.data_ptr(), dY.data_ptr())
                assert st.variant == PATCH
                images.add(st.patch)
                op(stream)
                torch.cuda.synchronize()
                np.testing.assert_array_equal(dY.cpu().numpy().view(np.uint16), ref.view(np.uint16), err_msg="%d x %d" % (Bn, H))
                first = first or (op, dX, dY, ref)
        sizes.append(held())
        print("round", rnd, "images", len(images), "bytes, buffers", sizes[-1], flush=True)
    assert len(images) == 16 and sizes[0] == sizes[1]
    one = 2 * w["nnzb"] * V  # the values alone; an image adds offsets, sources and padding
    assert sizes[0][0] <= 16 * (2 * one + 64 * 1024), sizes
    op, _, dY, ref = first
    dY.fill_(float("nan"))
    op(stream)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(dY.cpu().numpy().view(np.uint16), ref.view(np.uint16))
    f.release_scratch()
    assert held() == (0, 0)


def test_requests_for_shapes_beyond_those_held(torch_gpu):
    """All images taken: an explicit request that none of them suits says so (and leaves the others alone); the library takes a
    plane form; released, the filter takes the patch form again."""
    torch = torch_gpu
    C, F, V = 24, 64, 16
    w = P.make_weight(F, 9 * C, V, 0.3, True, 3, integer=True)
    f = P.upload_weight(w, 3, 3, C, cls=S.BlockwiseSpFilter)
    t = torch.zeros(64 * 80 * 80 * 64, dtype=torch.float16, device="cuda")
    images = set()
    for H in range(4, 70):
        for Bn, stride in ((1, 1), (3, 2), (16, 1), (1, 2), (6, 1), (16, 2)):
            images.add(S.SpconvBlockwiseOp().initialize(f, Bn, H, H, stride, t.data_ptr(), t.data_ptr()).patch)
    assert len(images) == 16 and None not in images
    # at stride 3 neighbouring positions lie 3 apart: another foot than any patch at strides 1 and 2
    refused = S.SpconvBlockwiseOp(PATCH)
    with pytest.raises(S.capi.ShflbwError) as e:
        refused.initialize(f, 2, 30, 30, 3, t.data_ptr(), t.data_ptr())
    assert e.value.status == S.capi.ERR_CAPACITY and "16 images" in str(e.value)
    assert S.SpconvBlockwiseOp().initialize(f, 2, 30, 30, 3, t.data_ptr(), t.data_ptr()).variant == 0
    f.release_scratch()
    assert S.SpconvBlockwiseOp().initialize(f, 2, 30, 30, 3, t.data_ptr(), t.data_ptr()).variant == PATCH
