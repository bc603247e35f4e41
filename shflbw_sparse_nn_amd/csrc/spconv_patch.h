// Launch-side description of the patch form of the convolution (host + device shared): one launch over NHWC tensors, a
// workgroup keeps the input patch its output pixels read in LDS, channel-major.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "kernel_common.h"

namespace shflbw {

// How a convolution is cut into workgroups.  Output positions are taken in blocks of tile_h x tile_w (at most
// 16 or 8) per image; four blocks ("units", any image, any place) make a column tile: column 4 p + u of the GEMM tile is
// position p of unit u.  The four units of a position lie side by side in LDS (8 bytes), which is what one lane of
// the transposing LDS read supplies, so a tap is a plain offset whatever the stride, the batch and the alignment.
struct ConvPatchPlan {
    int valid;            // some patch fits the LDS ...
    int col_blocks;       // 32-column blocks of a tile: 2 (16 positions x 4 units) or 1 (8 positions)
    int waves;            // waves of a workgroup
    int tile_h, tile_w;   // output positions of a unit
    int row_len;          // GEMM positions per tile row (>= tile_w; the surplus positions are no pixels)
    int blocks_w, blocks_hw, units;
    int step_h, step_w;   // patch positions between neighbouring output positions
    int patch_w, npos;    // columns and positions of the input patch of a unit
    int pitch;            // LDS bytes of one channel: 8 per position, an odd multiple of 8
    int groups, ksplit;   // waves = groups (rows) x ksplit (parts of the kept columns, a power of two: 1 << kshift)
    int kshift;
    int panels_per_wave;  // row units one wave computes one after the other
    int rows_wg, chunks;  // filters of a workgroup, workgroups per column tile
    int jobs, jobs_per_xcd;
    int H, W, Ho, Wo, stride, pad_h, pad_w; // extents as the kernel walks them (a 1 x 1 filter at stride 1: one row)
    int skip;             // stride wider than the filter in some direction
    unsigned in_bytes;
    unsigned touch_bytes, touch_step; // last byte of the filter image a workgroup brings into the L2; bytes one round of an XCD's threads covers
    int lds_bytes;
    unsigned magic_bhw, magic_bw, magic_pw, magic_row, magic_chunks, magic_pg;
    int preferred;        // ... and is estimated faster than the plane forms
    int slack;            // LDS bytes behind the row of zeros that columns without a pixel may touch
    int deep;             // 1: the kernel with more batches in flight, CONV_PATCH_WIDE: with all filters in a workgroup (see g_patch)
};

// What the plan depends on.
struct ConvPatchProblem {
    int V, F, C, R, S;
    double kept_per_panel; // kept columns of a row panel on average
    int permuted;          // rows of the filter are permuted
    int B, H, W, Ho, Wo, stride, cus;
};
// What the order of a filter image depends on: the patch as the LDS reads walk it.
struct ConvPatchShape {
    int pitch, patch_w;
    uint32_t foot; // bank pairs that the positions one pass of a transposing read touches lie in, for a row that starts in pair 0
    bool operator==(const ConvPatchShape& o) const { return pitch == o.pitch && patch_w == o.patch_w && foot == o.foot; }
};
ConvPatchShape conv_patch_shape(int rows, const ConvPatchPlan& p);
// rows of one pass of a transposing read: four of 8 positions, for row units of 16 eight of 4
inline int conv_patch_group(int rows) { return rows == 16 ? 8 : 4; }

// Fills `plan`; false when no patch fits the LDS (with `held`: none of these shapes) or the sizes leave 32-bit indexes.
// `wide_cuts` false: the plan without the wide kernels, which a check holds the other one against.
bool conv_patch_plan(const ConvPatchProblem& q, ConvPatchPlan* plan, const std::vector<ConvPatchShape>* held = nullptr, bool wide_cuts = true);

// Order of the kept columns of a row panel that keeps the LDS reads of a group of rows apart (see the definition).
struct ConvPatchOrder {
    ConvPatchOrder(uint32_t foot, int group);
    // pair_of: start pairs of the kept columns; `order` becomes their order, whole groups of `group` at a time
    void of(const std::vector<int>& pair_of, std::vector<int>& order) const;

private:
    uint32_t foot;
    int group;
    std::vector<std::vector<int>> tilings; // up to three exact ones, as shifts
    uint32_t touching(uint32_t set) const;
    void find_tilings(std::vector<int>& shifts, uint32_t used);
};

struct ConvPatchArgs {
    ConvPatchPlan p;
    int C, F, R, S;
    const half_t* in;
    half_t* out;
    // the filter as this form reads it: row units (a row panel; two for block height 128) of batches of 32 slots
    const half8_t* packedA;        // per batch the A fragments in register order
    const int* first_batch;        // per row unit its first batch, and the number of batches behind the last unit
    const unsigned short* offs;    // per batch the LDS offsets (in 8 bytes) of channel row and tap, in the order the lanes load them
    const unsigned short* dst;     // per stored row: its place among the staged rows of its workgroup
    const int* filt;               // per chunk and place: the filter (used when not dense)
    int dense;                     // the filters of a chunk are consecutive in the output
    int streams;                   // ... and leave by streaming stores (conv_patch_streams)
};

// Outputs from 60 MB on are streamed where the filters of a workgroup are consecutive; smaller ones, also three of them in turn,
// stay in the Infinity Cache and are written through.  1 x 1 on 64 channels, 56 x 56, us through / streamed: 16 -> 256 filters (26 MB)
// 9.2 / 9.3, 32 images -> 240 (48 MB) 25.3 / 26.3, 32 -> 256 (51 MB) 15.0 / 15.0, 64 -> 160 (64 MB) 35.6 / 31.6, 44 -> 256 (71 MB) 21.6 / 17.2, 48 -> 240
// (72 MB) 41.2 / 33.9, 64 -> 256 (103 MB) 36.0 / 25.0, 64 -> 304 (122 MB) 122 / 101.  (Ordinary stores: 25.1 for the 71 MB, 36.8 for the 103.)
inline bool conv_patch_streams(size_t out_bytes) { return out_bytes >= 60u << 20; }

// Packs the A fragments of `batches` batches from the weight's values (kept vectors one behind the other).  src: per batch and
// slot the row unit's part of a kept vector, as a multiple of `rows` values; -1: zeros (a padding slot).
hipError_t launch_patch_pack(const half_t* values, const int* src, half8_t* packedA, int rows, size_t batches, hipStream_t stream);

struct ConvPatchKernel {
    int RW, col_blocks, waves, deep;
    int per_cu; // workgroups of it the registers of a compute unit hold
    int ring, items; // batches a wave keeps in flight, patch items a thread keeps in flight
    int units;       // row units a wave may compute one after the other
    hipError_t (*launch)(const ConvPatchArgs&, hipStream_t);
    hipError_t (*prepare)();
};
const ConvPatchKernel* conv_patch_kernel(int rows, int col_blocks, int waves, int deep);

constexpr int CONV_PATCH_LDS_MAX = 160 * 1024;
constexpr int CONV_PATCH_SLACK = 256;       // least LDS bytes behind the row of zeros
constexpr int CONV_PATCH_TAIL_BATCHES = 8;  // batches of padding behind the last one: waves fetch ahead of their end
inline int conv_patch_unit_rows(int V) { return V == 128 ? 64 : V; }
constexpr int conv_patch_units(int rows) { return 64 / rows; } // row units of a wave but in the wide kernels
constexpr int CONV_PATCH_WIDE = 2;

} // namespace shflbw
