// The batch-innermost convolution that gathers from the input itself, in every cut that the library's choice knows and not only
// those that it takes at these sizes: the state's SpMM variant is set to each one that has a kernel.  Integer data, so every sum is
// exact and a result is the rounded oracle value or wrong.
#include "block_sparse/cuda_array.h"
#include "block_sparse/spconv/spconv_op.h"
#include "csrc/spconv_launch.h"
#include "oracle_reference.h"

struct Layer {
    int panels, B, H, W, C, R, S, stride;
    float density;
    bool permuted;
    int only_height; // block height it is run at, 0: all
};

// a lane's 8 images, tiles that end in mid-position, taps outside on every side; N is no multiple of any tile width
static const Layer layers[] = {
    {2, 8, 5, 9, 12, 3, 3, 1, 0.5f, true, 0},
    {3, 40, 13, 7, 5, 5, 5, 2, 0.3f, false, 0},
    {1, 8, 4, 40, 3, 1, 31, 1, 0.5f, true, 0},   // as many taps as a lane keeps bits for
    {2, 104, 15, 3, 70, 1, 1, 2, 0.9f, true, 0},
    {4, 24, 6, 11, 10, 2, 4, 3, 0.01f, false, 0}, // even extents, panels that keep next to nothing
    {2, 8, 6, 7, 64, 5, 5, 1, 0.5f, true, 0},     // panels of 25 stages, longer than every ring
    {2, 16, 1, 57, 33, 3, 3, 1, 0.7f, true, 0},   // one row
    {12, 8, 41, 39, 9, 3, 3, 1, 0.4f, true, 0},   // more tiles of every width than the chip holds workgroups
    {4, 128, 14, 14, 256, 3, 3, 1, 0.1f, true, 64}, // the reference's test layer
};

int main()
{
    int failures = 0;
    for (int V : {16, 32, 64, 128})
        for (const Layer& l : layers) {
            if (l.only_height && l.only_height != V) continue;
            BlockwiseSpFilter<half> f;
            f.init_random(l.panels * V, l.R, l.S, l.C, V, 1, l.density, l.permuted, 2021u);
            f.fmap_layout = fmap_batch_first;
            f.transform_and_sync_device();
            CudaRandomArray<half> in;
            CudaZerosArray<half> out;
            in.initialize(l.C * l.H * l.W * l.B);
            out.initialize(f.F * l.H * l.W * l.B);
            std::vector<float> ref;
            oracle_reference_batch_first<half>(f, l.B, l.H, l.W, l.stride, in.host_array, ref);
            shflbw_spconv_state state;
            SHFLBW_CHECK(shflbw_spconv_init_chwb(&state, f.handle(), l.B, l.H, l.W, l.stride, in.device_ptr, out.device_ptr));
            if (state.planes) {
                printf("block height %d: the layer runs over planes Failed\n", V);
                return EXIT_FAILURE;
            }
            for (int i = 0; i < shflbw_spmm_variant_count(V); i++) {
                const char* name = shflbw_spmm_variant_name(V, i);
                const shflbw::ConvTapsKernel* k = shflbw::conv_taps_kernel(name);
                if (!k) continue;
                printf("%s: %d x %d x %d x %d -> %d, %d x %d, stride %d", name, l.B, l.H, l.W, l.C, f.F, l.R, l.S, l.stride);
                fflush(stdout);
                HIP_CHECK(k->prepare());
                HIP_CHECK(hipMemset(out.device_ptr, 0xff, sizeof(half) * out.size)); // NaN
                state.spmm.variant = i;
                SHFLBW_CHECK(shflbw_spconv_exec(&state, nullptr));
                HIP_CHECK(hipDeviceSynchronize());
                out.sync_host();
                size_t bad = 0;
                for (size_t e = 0; e < ref.size(); e++)
                    bad += !(static_cast<float>(out.host_array[e]) == static_cast<float>(static_cast<half>(ref[e])));
                printf(bad ? " Failed (%zu values)\n" : " Passed\n", bad);
                failures += bad != 0;
            }
        }
    printf(failures ? "FAILED %d failure(s)\n" : "ALL PASSED\n", failures);
    return failures ? EXIT_FAILURE : EXIT_SUCCESS;
}
