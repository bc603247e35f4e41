// Device side of the C ABI: uploads of the weight images and the SpMM / SpConv
// init + exec entry points.  Reference: block_sparse/spmm/blockwise_format.h:230-266
// (upload), block_sparse/spmm/blockwise_op.h:81-215 and
// block_sparse/spconv/blockwise_op.h:79-193 (init / exec).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "shflbw.h"
#include "spconv_launch.h"
#include "spmm_launch.h"
#include "weight_internal.h"

namespace shflbw {

#define SHFLBW_HIP_TRY(expr)                                                                            \
    do {                                                                                                \
        hipError_t e_ = (expr);                                                                         \
        if (e_ != hipSuccess) {                                                                         \
            set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__, __LINE__);       \
            return SHFLBW_ERR_HIP;                                                                      \
        }                                                                                               \
    } while (0)

static void release_conv_scratch(shflbw_weight* w);

void clear_device(shflbw_weight* w)
{
    if (w->d_image) (void)hipFree(w->d_image);
    for (void** b : {&w->d_image, &w->d_meta, &w->d_values, &w->d_group_ptr, &w->d_packed_indices, &w->d_packed_indices_pm,
                     &w->d_packed_values, &w->d_packed_slab})
        *b = nullptr;
    release_conv_scratch(w);
}

// frees every device buffer the convolution inits of this weight allocated (the caller holds scratch_lock or owns w)
void release_conv_scratch(shflbw_weight* w)
{
    for (auto& e : w->conv_ids)
        if (e.ptr) (void)hipFree(e.ptr);
    for (auto& e : w->conv_bulk)
        if (e.ptr) (void)hipFree(e.ptr);
    for (auto& e : w->patch_images)
        if (e.ptr) (void)hipFree(e.ptr);
    for (auto& e : w->patch_places)
        if (e.ptr) (void)hipFree(e.ptr);
    w->conv_ids.clear();
    w->conv_bulk.clear();
    w->patch_images.clear();
    w->patch_places.clear();
    w->patch_geometries.clear();
}

// One allocation and one copy for all arrays of a weight (seven of each cost more than packing a small weight).
int upload(shflbw_weight* w)
{
    struct Part {
        void** dst;
        const void* src;
        size_t bytes, at;
    } parts[] = {
        {&w->d_meta, w->meta_h.data(), w->meta_h.size() * sizeof(int), 0},
        {&w->d_values, w->values.data(), w->values.size() * sizeof(uint16_t), 0},
        {&w->d_group_ptr, w->panel_desc.data(), w->panel_desc.size() * sizeof(int), 0},
        {&w->d_packed_indices, w->packed_indices.data(), w->packed_indices.size() * sizeof(int), 0},
        {&w->d_packed_indices_pm, w->packed_indices_pm.data(), w->packed_indices_pm.size() * sizeof(int), 0},
        {&w->d_packed_values, w->packed_values.data(), w->packed_values.size() * sizeof(uint16_t), 0},
        {&w->d_packed_slab, w->packed_slab.data(), w->packed_slab.size() * sizeof(int), 0},
    };
    size_t total = 0;
    for (Part& p : parts) {
        p.at = total;
        total += (p.bytes + 16 + 255) / 256 * 256; // zero-length arrays (an empty matrix) still get a valid pointer
    }
    std::unique_ptr<unsigned char[]> host(new unsigned char[total]);
    for (Part& p : parts)
        if (p.bytes) memcpy(host.get() + p.at, p.src, p.bytes);
    SHFLBW_HIP_TRY(hipMalloc(&w->d_image, total));
    for (Part& p : parts) *p.dst = (char*)w->d_image + p.at;
    if (hipMemcpy(w->d_image, host.get(), total, hipMemcpyHostToDevice) != hipSuccess) {
        clear_device(w);
        set_error("sync_device: cannot upload %zu bytes", total);
        return SHFLBW_ERR_HIP;
    }
    return SHFLBW_OK;
}

// compute units of the current device, looked up once per device
static int device_compute_units()
{
    static std::atomic<int> cached[64]; // two threads may look the same number up at once
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int n = cached[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

// The variants of a block height lie side by side in the table.  Every initialisation and launch looks one up: the ranges
// are found once.
static const SpmmVariant* find_spmm_variant(int brow, int variant, int* n_for_brow)
{
    struct Ranges {
        const SpmmVariant* first[4] = {};
        int n[4] = {};
        static int of(int brow) { return brow == 16 ? 0 : brow == 32 ? 1 : brow == 64 ? 2 : brow == 128 ? 3 : -1; }
        Ranges()
        {
            int count = 0;
            const SpmmVariant* all = spmm_variants(&count);
            for (int i = 0; i < count; i++) {
                const int r = of(all[i].V);
                if (n[r]++ == 0) first[r] = &all[i];
            }
        }
    };
    static const Ranges ranges;
    const int r = Ranges::of(brow), n = r < 0 ? 0 : ranges.n[r];
    if (n_for_brow) *n_for_brow = n;
    return variant >= 0 && variant < n ? ranges.first[r] + variant : nullptr;
}

static const SpconvVariant* find_spconv_variant(int brow, int variant, int* n_for_brow)
{
    int count = 0;
    const SpconvVariant* all = spconv_variants(&count);
    const SpconvVariant* hit = nullptr;
    int seen = 0;
    for (int i = 0; i < count; i++) {
        if (all[i].V != brow) continue;
        if (seen == variant) hit = &all[i];
        seen++;
    }
    if (n_for_brow) *n_for_brow = seen;
    return hit;
}

static bool spmm_variant_splits(const SpmmVariant* v) { return v && strncmp(v->name, "split", 5) == 0; }
// the persistent role-split variants ("ws..." names) form gather addresses from 32-bit byte offsets; the split form is for
// few columns and holds to the same bound
static bool spmm_variant_offsets32(const SpmmVariant* v) { return v && (v->name[0] == 'w' || spmm_variant_splits(v)); }

// Tile choice when the caller does not force one: the variant with the least estimated time.  The weights are us, fitted to 13 860 problems
// (profiles/spmm_estimate_fit.py draws, times and fits them: 64-65536 rows, 64-16384 columns of A, 8-131072 of B, densities of 0.02-0.5,
// up to four times the work of 8192 x 4096 x 16384 at block height 128, a fifth of them with a C term; every variant of their block
// height timed over three sets of operands in turn), so that the variant with the least estimate takes little longer than the
// fastest one; no weight says what its part costs by itself.  Over 4620 problems drawn and timed after the fit the choice takes
// 1.009 times the fastest variant's time (geometric mean), more than 1.1 times on 61.
// Before: a least-squares fit to 1390 problems up to the work of the largest case, with one D term however D is stored and the
// mean number of tiles for long panels that two workgroups of a compute unit share: 1.021 times, more than 1.1 times on 323.  It took
// narrow tiles where D is large (12416 x 69 x 63096, block height 128, density 0.05: 794 us, now 553; 5952 x 744 x 64552, 64: 340 and 299) and where
// long panels fill a few compute units twice (5472 x 3207 x 368, 32, 0.37: 19.2 and 15.7).  The lines drawn by hand before that
// (bounds on tiles, columns and kept vectors) take 1.09 times on average and 2.8 at worst, above all for many panels over few
// columns on 512-column tiles (29632 x 761 x 64, density 0.47, block height 64: 16.1 us; 128-column tiles 7.0).
//
//  role-split: base + tiles of a compute unit * (tile + stage * stages of 32 kept vectors) + D.  The tiles of a compute unit are
//    their number rounded up.  Where two workgroups share one, a second tile beside the first counts as second.tile and second.stage,
//    its presence costs second.start, and per tile, other than per stage, the mean number counts;
//  slab: base + rounds * (slab + K / 1000 * row + panels of a wave * (panel + batches of 32 vectors * batch)) + D;
//  split: base + rounds * (tile + steps of a wave * (step + (64 columns: wide_step))) + D;
//  D: its bytes at 5 TB/s times the weight of the way it is stored (by StoreMode), and what exceeds the Infinity Cache times `beyond`.
//  With a C term c * (C at 5 TB/s) and c_tile for every tile (round of the split form, panel of a wave) more.
struct StoreWeights {
    float by_mode[3], beyond;
    double of(StoreMode mode, double t_d) const { return by_mode[mode] * t_d + beyond * std::max(0.0, t_d - 53.7); }
};
struct SecondTile {
    float start, tile, stage;
    double tiles(double mean) const { return mean <= 2 ? 1 + (mean - 1) * tile : mean / 2 * (1 + tile); }
    double stages(double n) const { return std::floor(n / 2) * (1 + stage) + n - 2 * std::floor(n / 2); }
};
struct RoleSplitEstimate {
    const char* name;
    float base, tile, stage;
    StoreWeights d;
    float c, c_tile;
    SecondTile second; // variants with two workgroups per compute unit only
};
struct SlabEstimate {
    const char* name;
    float base, slab, row, panel, batch;
    StoreWeights d;
    float c, c_panel;
};
struct SplitEstimate {
    const char* name;
    float base, tile, step, wide_step, d, c, c_round;
};
static const RoleSplitEstimate g_role_split_estimates[] = {
    {"ws16x128x4c4p_k32_s4", 2.04f, 0.747f, 0.317f, {1.05f, 0.578f, 0.f, 0.f}, 0.661f, 0.298f},
    {"ws16x64x4c4p_k32_s4", 1.74f, 0.637f, 0.215f, {0.f, 0.0566f, 0.f, 0.0226f}, 0.f, 0.286f, {0.286f, 0.922f, 0.619f}},
    {"ws16x64x2c4p_k32_s6", 2.12f, 0.396f, 0.161f, {0.f, 0.113f, 0.f, 0.f}, 0.421f, 0.176f, {0.0802f, 1.49f, 0.402f}},
    {"ws32x128x4c4p_k32_s4", 2.06f, 0.893f, 0.364f, {0.941f, 1.11f, 0.729f, 0.f}, 0.726f, 0.722f},
    {"ws32x64x4c4p_k32_s3", 1.35f, 0.871f, 0.429f, {0.202f, 0.638f, 0.f, 0.227f}, 0.409f, 0.617f, {0.296f, 0.429f, 0.343f}},
    {"ws32x64x4c4p_k32_s6", 1.32f, 1.38f, 0.22f, {0.0374f, 0.0822f, 0.f, 0.f}, 0.235f, 0.524f},
    {"ws32x32x4c4p_k32_s6", 1.56f, 0.948f, 0.165f, {0.f, 0.23f, 0.f, 0.28f}, 0.487f, 0.311f, {0.193f, 0.28f, 0.569f}},
    {"ws64x128x4c4p_k32_s4", 1.67f, 1.99f, 0.478f, {0.659f, 0.718f, 0.461f, 0.228f}, 0.599f, 1.49f},
    {"ws64x64x4c4p_k32_s3", 0.444f, 1.38f, 0.586f, {0.635f, 0.899f, 0.169f, 0.586f}, 0.657f, 1.49f, {0.838f, 0.0779f, 0.f}},
    {"ws64x64x4c4p_k32_s6", 1.49f, 1.4f, 0.295f, {0.379f, 0.636f, 0.129f, 0.281f}, 0.271f, 1.36f},
    {"ws64x32x4c4p_k32_s4", 1.32f, 0.44f, 0.247f, {0.677f, 1.03f, 0.591f, 0.594f}, 0.211f, 0.928f, {0.758f, 0.624f, 0.419f}},
    {"ws64x32x4c4p_k32_s6", 1.02f, 1.48f, 0.207f, {0.f, 0.f, 0.f, 0.0376f}, 0.00714f, 0.764f},
    {"ws128x64x4c4p_k32_s6", 0.27f, 3.63f, 0.415f, {0.251f, 0.00972f, 0.f, 0.55f}, 0.543f, 1.14f},
    {"ws128x32x4c4p_k32_s4", 0.f, 2.74f, 0.297f, {0.515f, 0.339f, 0.339f, 0.896f}, 1.03f, 0.923f, {0.967f, 0.0828f, 0.816f}},
    {"ws128x32x4c4p_k32_s6", 0.694f, 2.52f, 0.268f, {0.372f, 0.471f, 0.0712f, 0.f}, 0.296f, 1.13f},
};
static const SlabEstimate g_slab_estimates[] = {
    {"slab16x64", 1.52f, 1.19f, 2.22f, 0.f, 0.168f, {0.894f, 1.05f, 0.604f, 0.0739f}, 0.0722f, 0.624f},
    {"slab32x64", 0.f, 2.91f, 1.98f, 0.211f, 0.235f, {0.89f, 0.794f, 0.83f, 0.376f}, 0.374f, 0.848f},
};
static const SplitEstimate g_split_estimates[] = {
    {"split16x32", 0.78f, 1.57f, 0.843f, 0.2f, 3.67f, 0.f, 0.205f},
    {"split32x32", 1.03f, 2.2f, 0.541f, 0.306f, 0.579f, 0.8f, 0.263f},
    {"split64x32", 1.02f, 2.07f, 0.634f, 0.502f, 0.642f, 0.f, 0.608f},
    {"split128x32", 0.333f, 1.5f, 0.775f, 0.798f, 1.68f, 1.12f, 0.501f},
};

static StoreMode result_store_mode(const void* D, int rows, int ldd, size_t others, bool narrow, bool read_back);
// role-split tiles of 128 columns, but for block height 16, are stored by half lines (ws_consumer)
static bool stores_half_lines(int brow, int tile_cols) { return brow != 16 && tile_cols == 128; }

// What an estimate depends on.
struct SpmmProblem {
    const shflbw_weight* w;
    int N, X, cus;
    double vectors; // kept per panel
    double t_d;     // D (and C) at 5 TB/s
    bool residual;
    size_t others;  // bytes of B and C
};

static double estimate(const SpmmVariant& v, const RoleSplitEstimate& e, const SpmmProblem& q)
{
    const double mean = (double)q.X * ((q.N + v.BN - 1) / v.BN) / q.cus, n = std::ceil(mean);
    const bool two = v.per_cu == 2;
    const double tiles = two ? e.second.tiles(std::max(1.0, mean)) : n, stages = two ? e.second.stages(n) : n;
    const double t = e.base + e.tile * tiles + e.stage * (q.vectors / 32 + 0.5) * stages + (two && n >= 2 ? e.second.start : 0.f) +
                     e.d.of(result_store_mode(nullptr, q.w->nrow, q.N, q.others, stores_half_lines(q.w->brow, v.BN), false), q.t_d);
    return q.residual ? t + e.c * q.t_d + e.c_tile * tiles : t;
}

static double estimate(const SpmmVariant& v, const SlabEstimate& e, const SpmmProblem& q)
{
    const SlabDeal s = slab_deal(q.w->brow, q.X, q.w->ncol, (int)(q.w->packed_indices.size() / 64), (q.N + v.BN - 1) / v.BN, q.cus / 8 * 8);
    const double panels = (double)s.rounds * s.wave_panels;
    const double t = e.base + s.rounds * (e.slab + e.row * q.w->ncol / 1000) + panels * (e.panel + e.batch * 2 * std::ceil(q.vectors / 64)) +
                     e.d.of(slab_store_mode(nullptr, q.w->nrow, q.N, q.others), q.t_d);
    return q.residual ? t + e.c * q.t_d + e.c_panel * panels : t;
}

static double estimate(const SpmmVariant&, const SplitEstimate& e, const SpmmProblem& q) // as launch_split cuts it
{
    const bool v16 = q.w->brow == 16;
    const double blocks = q.w->nrow / (v16 ? 16 : 32);
    const bool wide = !v16 && q.N > 32 && blocks * ((q.N + 31) / 32) > q.cus;
    const double grid = std::ceil(blocks / 8) * 8 * (wide ? (q.N + 63) / 64 : (q.N + 31) / 32);
    const int waves = grid <= q.cus ? 16 : 8;
    const double steps = q.vectors / (v16 ? 32 : 16) / waves + 0.5;
    const double mean = std::max(1.0, grid / (waves == 16 ? q.cus : 2 * q.cus)), rounds = 0.5 * (mean + std::ceil(mean));
    const double t = e.base + rounds * (e.tile + (e.step + (wide ? e.wide_step : 0.f)) * steps) + e.d * q.t_d;
    return q.residual ? t + e.c * q.t_d + e.c_round * rounds : t;
}

// `spmm` false: what is multiplied are the planes of a convolution, which only the variants that gather rows by id can walk.
static int auto_spmm_variant(const shflbw_weight* w, int N, bool spmm, bool residual, int compute_units)
{
    struct Candidates { // of the four block heights, found once
        struct One {
            const SpmmVariant* v;
            int number;
            const RoleSplitEstimate* role_split; // one of the three
            const SlabEstimate* slab;
            const SplitEstimate* split;
        };
        std::vector<One> of[4];
        Candidates()
        {
            for (int h = 0; h < 4; h++) {
                int count = 0;
                const SpmmVariant* all = find_spmm_variant(16 << h, 0, &count);
                for (int i = 0; i < count; i++) {
                    for (const RoleSplitEstimate& e : g_role_split_estimates)
                        if (strcmp(e.name, all[i].name) == 0) of[h].push_back({&all[i], i, &e, nullptr, nullptr});
                    for (const SlabEstimate& e : g_slab_estimates)
                        if (strcmp(e.name, all[i].name) == 0) of[h].push_back({&all[i], i, nullptr, &e, nullptr});
                    for (const SplitEstimate& e : g_split_estimates)
                        if (strcmp(e.name, all[i].name) == 0) of[h].push_back({&all[i], i, nullptr, nullptr, &e});
                }
            }
        }
    };
    static const Candidates candidates;
    const int h = w->brow == 16 ? 0 : w->brow == 32 ? 1 : w->brow == 64 ? 2 : w->brow == 128 ? 3 : -1;
    if (h < 0 || w->nrow <= 0) return 0;
    SpmmProblem q{w, N, w->nrow / w->brow, compute_units, 0, 2.0 * w->nrow * N / 5e6, residual, ((size_t)w->ncol + (residual ? w->nrow : 0)) * N * 2};
    q.vectors = (double)w->nnzb / q.X;
    int best = 0;
    double least = 0;
    for (const auto& c : candidates.of[h]) {
        if (!c.role_split && !spmm) continue;
        if (c.slab && (w->packed_slab.empty() || w->ncol > c.v->max_k)) continue;
        if (c.split && N > 1024) continue;
        const double t = c.role_split ? estimate(*c.v, *c.role_split, q) : c.slab ? estimate(*c.v, *c.slab, q) : estimate(*c.v, *c.split, q);
        if (least == 0 || t < least) least = t, best = c.number;
    }
    return best;
}

// Geometry of the plane form of a convolution and the layout of its device scratch.
struct PlaneForm {
    int PH, PW;     // rows and (padded to 8) columns of one phase plane
    int copies;     // 2 when some tap offset is odd (a second copy moved by one value keeps gathers aligned)
    long np;        // plane positions = columns of the SpMM in the middle
    long pitch;     // values per channel row of the plane tensor
    long rows;      // channel rows: copies * stride^2 * C
    size_t slots;   // padded kept-vector slots of the filter
    int Ho, Wo;
    size_t planes_bytes, dm_bytes, ids_bytes; // planes | result_fm, and (the entry point without allocation) | ids | ids_pm behind them
    size_t total_bytes() const { return planes_bytes + dm_bytes + 2 * ids_bytes; }
};

// `rows` channel rows of `pitch` values and a row of zeros behind them: within the 4 GiB of 32-bit byte offsets?
static bool planes_fit(long rows, long pitch) { return rows < 0x7fffffffL / pitch; }

static int plane_form_geometry(const shflbw_weight* f, int B, int H, int W, int stride, PlaneForm* g)
{
    const int s = stride, ph = f->R / 2, pw = f->S / 2;
    g->copies = (f->S - 1) / s >= 1 ? 2 : 1;
    if (s > 5 || g->copies * s * s > 32) {
        set_error("spconv: stride %d has too many phase planes for the plane form", s);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    g->PH = (H + 2 * ph + s - 1) / s;
    g->PW = ((W + 2 * pw + s - 1) / s + 7) / 8 * 8;
    g->np = (long)B * g->PH * g->PW;
    const long max_shift = (long)((f->R - 1) / s) * g->PW + (f->S - 1) / s; // largest tap offset
    g->pitch = (g->np + max_shift + 8 + 63) / 64 * 64;
    g->rows = (long)g->copies * s * s * f->C;
    if (g->np > 0x7fffffffL || !planes_fit(g->rows, g->pitch)) {
        set_error("spconv: problem too large for the plane form (%ld rows of %ld positions)", g->rows, g->pitch);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    auto up256 = [](size_t n) { return (n + 255) / 256 * 256; };
    g->slots = f->packed_indices.size();
    g->planes_bytes = up256((size_t)(g->rows + 1) * g->pitch * 2); // one more row: zeros, for the padding slots
    g->dm_bytes = up256((size_t)f->F * g->np * 2);
    g->ids_bytes = up256(g->slots * sizeof(int) + 64);
    g->Ho = (H + 2 * ph - f->R) / s + 1;
    g->Wo = (W + 2 * pw - f->S) / s + 1;
    return SHFLBW_OK;
}

// How the role-split kernels store D.  `others`: bytes of B and C.
//  * Rows that do not start at whole lines: every line is written in parts, by neighbouring store instructions, and each part
//    written through is a write of its own to the Infinity Cache, or to memory where that does not hold the line.  Merged in the L2
//    where it will not: where three such problems in turn, 3 * (B + C + D), do not fit its 256 MB.  Merged / through, 600 drawn
//    problems with D of 8 to 300 MB (955 pairs with a variant without C, 397 with): 0.92 by this rule, 6 pairs above 1.05; with
//    the line at D >= 24 MB, as before, 0.92 and 85, up to 1.22 (32 x 1184 x 279 x 13792, 33 MB, short panels: 9.8 us through, 12.0).
//    Narrow tiles, whose stores are half lines, from 24 MB on (0.88 below the other line).
//  * Whole lines: streamed from 96 MB on, if nothing reads D back at once; smaller results, also three of them in turn, stay in
//    the Infinity Cache.  us, through / streamed, density 0.1, block height 64, K = 1640 or 2048: 16384 x 1024 12.5 / 12.9 (33 MB),
//    6144 x 4096 30.8 / 30.3 (50 MB), 16384 x 2560 28.6 / 28.5, 16384 x 2816 34.3 / 33.0 (92 MB), 8192 x 6400 45 / 40, 8192 x 8192 58 / 50;
//    block height 128: 16384 x 2048 23.5 / 26.0 (67 MB), 16384 x 2816 35.3 / 37.1, 8192 x 6400 74 / 69, 4096 x 16384 65 / 52; 16:
//    16384 x 4096 110 / 89.  Merged: as written through for large D, 4096^3 21 / 25.
static StoreMode result_store_mode(const void* D, int rows, int ldd, size_t others, bool narrow, bool read_back)
{
    const size_t bytes = (size_t)rows * (size_t)ldd * 2;
    if ((((uintptr_t)D | ((uintptr_t)ldd * 2)) & 127) != 0)
        return bytes + others >= STORE_MERGE_BYTES || (narrow && bytes >= 24u << 20) ? STORE_MERGE : STORE_THROUGH;
    return bytes >= 96u << 20 && !read_back ? STORE_STREAM : STORE_THROUGH;
}

void fill_spmm_launch_args(const shflbw_spmm_state* state, int BN, SpmmLaunchArgs* out)
{
    SpmmLaunchArgs& a = *out;
    a.M = state->args.M;
    a.N = state->args.N;
    a.K = state->args.K;
    a.X = a.M / state->brow;
    a.magic_x = udiv_magic(a.X);
    a.n_tiles = 0;
    a.packedA = (const half8_t*)state->packed_values;
    a.kidx = state->packed_indices;
    a.kidx_pm = state->packed_indices_pm;
    a.slab_ids = state->packed_slab;
    a.slab_chunks = 1, a.slab_panels = a.X, a.slab_by_chunk = 0;
    a.groups = state->groups;
    a.half_panels = state->half_panels;
    a.panel_desc = state->panel_ptr;
    a.row_ids = state->args.A_row_indices;
    a.B = (const half_t*)state->args.B;
    a.ldb_bytes = state->ldb_bytes;
    a.zero_row = state->zero_row;
    a.C = (const half_t*)state->args.C;
    a.D = (half_t*)state->args.D;
    a.alpha = state->args.alpha;
    a.beta = state->args.beta;
    a.num_cus = device_compute_units();
    a.ldd = a.N;
    a.store_mode = result_store_mode(a.D, a.M, a.ldd, bytes_of_b_and_c(a), stores_half_lines(state->brow, BN),
                                     a.ldb_bytes != a.N * 2); // (planes: the layout kernel behind it reads D)
    a.dmap_row = a.dmap_valid = 0, a.dmap_magic = 0;
    // rows of B one column tile can touch: above about 2.5 MB they do not stay in the 4 MB L2 of an XCD
    // from one round of tiles to the next, and alternating the direction of the walk pays (measured:
    // +1 % at 2 MB, -4 % at 3 MB, -7 % at 4 MB, -13 % at 8 MB)
    a.alternate = (double)a.K * a.ldb_bytes * BN / (a.N > 0 ? a.N : 1) > 2.5 * 1024 * 1024;
}

} // namespace shflbw

using namespace shflbw;

extern "C" {

int shflbw_spmm_variant_count(int brow)
{
    int n = 0;
    find_spmm_variant(brow, 0, &n);
    return n;
}

const char* shflbw_spmm_variant_name(int brow, int variant)
{
    const SpmmVariant* v = find_spmm_variant(brow, variant, nullptr);
    return v ? v->name : "";
}

// `gather_only`: the caller will point the gather at something other than a K x N matrix (the planes of a
// convolution, ids rewritten as element offsets), which only the variants that gather rows by id can walk: the
// variants that hold all K rows of B in LDS are left out of the automatic choice and refused when forced.  There is no
// K x N matrix then, and its size bounds nothing: the caller keeps what its ids address below 4 GiB.
static int spmm_init_impl(shflbw_spmm_state* state, const shflbw_weight* w, int N, const void* B, const void* C, void* D,
                          float alpha, float beta, int variant, bool gather_only)
{
    if (!state) return SHFLBW_ERR_INVALID;
    memset(state, 0, sizeof(*state));
    if (!w || !B || !D) {
        set_error("spmm_init: null weight, B or D");
        return SHFLBW_ERR_INVALID;
    }
    if (!w->device_synced) { // assert at blockwise_op.h:87
        set_error("spmm_init: sparse matrix is not synced to device");
        return SHFLBW_ERR_STATE;
    }
    if (w->bcol != 1) { // assert at blockwise_op.h:86 (BK = 1)
        set_error("spmm_init: bcol must be 1 (got %d)", w->bcol);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    if (N <= 0 || (N % 8) != 0) {
        set_error("spmm_init: N must be a positive multiple of 8 (got %d)", N);
        return SHFLBW_ERR_SHAPE;
    }
    if (beta != 0.f && !C) {
        set_error("spmm_init: beta != 0 needs C");
        return SHFLBW_ERR_INVALID;
    }
    if (((uintptr_t)B | (uintptr_t)D | (uintptr_t)C) & 15) {
        set_error("spmm_init: B, C and D must be 16-byte aligned");
        return SHFLBW_ERR_INVALID;
    }
    const int X = w->nrow / w->brow, compute_units = device_compute_units();
    // the role-split kernels address the rows of B with 32-bit byte offsets
    const bool wide_b =
        !gather_only && (unsigned long long)w->ncol * (unsigned long long)N * 2ull + (unsigned long long)N * 2ull > 0xffffffffull;
    if (variant < 0) {
        variant = auto_spmm_variant(w, N, !gather_only, beta != 0.f, compute_units);
        if (wide_b) { // first variant of this block size with 64-bit addressing (block height 16 has none: refused below)
            int n = 0;
            find_spmm_variant(w->brow, variant = 0, &n);
            for (int i = 0; i < n; i++)
                if (const SpmmVariant* c = find_spmm_variant(w->brow, i, nullptr); !spmm_variant_offsets32(c) && c->max_k == 0) {
                    variant = i;
                    break;
                }
        }
    }
    const SpmmVariant* v = find_spmm_variant(w->brow, variant, nullptr);
    if (!v) {
        set_error("spmm_init: no tile variant %d for block size %d", variant, w->brow);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    if (v->max_k > 0 && gather_only) {
        set_error("spmm_init: tile variant %s holds the rows of B in LDS and cannot walk the planes of a convolution", v->name);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    if (v->max_k > 0 && (w->ncol > v->max_k || w->packed_slab.empty())) {
        set_error("spmm_init: tile variant %s holds all rows of B in LDS: at most %d columns of A (got %d)", v->name,
                  v->max_k, w->ncol);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    if (wide_b && spmm_variant_offsets32(v)) {
        set_error("spmm_init: B (%d x %d fp16) exceeds the 4 GiB the tile variant %s can address", w->ncol, N, v->name);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    SpmmLaunchArgs la;
    la.M = w->nrow, la.N = N, la.X = X, la.num_cus = compute_units;
    SHFLBW_HIP_TRY(v->prepare(la));

    shflbw_device_ref ref;
    shflbw_weight_device_ref(w, &ref);
    state->args.M = w->nrow;
    state->args.N = N;
    state->args.K = w->ncol;
    state->args.A_values = ref.csb_values;
    state->args.B = B;
    state->args.C = C;
    state->args.D = D;
    state->args.A_bsr_indptr = ref.csb_indptr;
    state->args.A_bsr_indices = ref.csb_indices;
    state->args.A_row_indices = ref.row_permute_ids;
    state->args.alpha = alpha;
    state->args.beta = beta;
    state->packed_values = w->d_packed_values;
    state->packed_indices = (const int*)w->d_packed_indices;
    state->packed_indices_pm = (const int*)w->d_packed_indices_pm;
    state->packed_slab = w->packed_slab.empty() ? nullptr : (const int*)w->d_packed_slab;
    state->groups = (int)(w->packed_indices.size() / 64);
    state->half_panels = w->half_panels;
    state->panel_ptr = (const int*)w->d_group_ptr;
    state->brow = w->brow;
    state->ldb_bytes = N * 2;
    state->zero_row = spmm_zero_row();
    if (!state->zero_row) {
        set_error("spmm_init: cannot look up the library's row of zeros on this device");
        return SHFLBW_ERR_HIP;
    }
    state->variant = variant;
    state->shared_mem_size = (size_t)v->lds_bytes;
    state->grid_dim[0] = (unsigned)(X * ((N + v->BN - 1) / v->BN));
    state->grid_dim[1] = state->grid_dim[2] = 1;
    state->block_dim[0] = (unsigned)v->threads;
    state->block_dim[1] = state->block_dim[2] = 1;
    state->init_success = 1;
    return SHFLBW_OK;
}

int shflbw_spmm_init_variant(shflbw_spmm_state* state, const shflbw_weight* w, int N, const void* B, const void* C,
                             void* D, float alpha, float beta, int variant)
{
    return spmm_init_impl(state, w, N, B, C, D, alpha, beta, variant, false);
}

int shflbw_spmm_init(shflbw_spmm_state* state, const shflbw_weight* w, int N, const void* B, const void* C, void* D,
                     float alpha, float beta)
{
    return shflbw_spmm_init_variant(state, w, N, B, C, D, alpha, beta, -1);
}

int shflbw_spmm_exec(const shflbw_spmm_state* state, void* stream)
{
    if (!state || !state->init_success) {
        set_error("spmm_exec: state was not initialised successfully");
        return SHFLBW_ERR_STATE;
    }
    const SpmmVariant* v = find_spmm_variant(state->brow, state->variant, nullptr);
    if (!v) return SHFLBW_ERR_UNSUPPORTED;
    SpmmLaunchArgs a;
    fill_spmm_launch_args(state, v->BN, &a);
    if (a.X == 0) return SHFLBW_OK;
    hipError_t e = v->launch(a, (hipStream_t)stream);
    if (e != hipSuccess) {
        set_error("spmm_exec: launch failed: %s", hipGetErrorString(e));
        return SHFLBW_ERR_HIP;
    }
    return SHFLBW_OK;
}


int shflbw_spconv_init(shflbw_spconv_state* state, const shflbw_weight* f, int B, int H, int W, int stride,
                       const void* IFMap, void* OFMap)
{
    return shflbw_spconv_init_variant(state, f, B, H, W, stride, IFMap, OFMap, -1);
}

} // extern "C"

namespace {

// forms of the convolution (shflbw_spconv_variant_name)
enum ConvForm { FORM_PLANES = 0, FORM_DIRECT = 1, FORM_BPLANES = 2, FORM_FUSED = 3, FORM_CHWB = 4, FORM_PATCH = 5, FORM_COUNT = 6 };

// Argument checks of a convolution and every field of the state that does not depend on device scratch.
int spconv_fill_state(shflbw_spconv_state* state, const shflbw_weight* f, int B, int H, int W, int stride,
                      const void* IFMap, void* OFMap, int variant)
{
    if (!state) return SHFLBW_ERR_INVALID;
    memset(state, 0, sizeof(*state));
    if (!f || !IFMap || !OFMap) {
        set_error("spconv_init: null filter, IFMap or OFMap");
        return SHFLBW_ERR_INVALID;
    }
    if (!f->device_synced) { // assert at spconv/blockwise_op.h:83
        set_error("spconv_init: sparse filter is not synced to device");
        return SHFLBW_ERR_STATE;
    }
    if (f->R <= 0) {
        set_error("spconv_init: weight has no filter view (use shflbw_filter_init_random or pass R,S,C to shflbw_weight_set)");
        return SHFLBW_ERR_STATE;
    }
    if (f->bcol != 1) {
        set_error("spconv_init: bcol must be 1 (got %d)", f->bcol);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    if (B <= 0 || H <= 0 || W <= 0 || stride <= 0) {
        set_error("spconv_init: non-positive B, H, W or stride");
        return SHFLBW_ERR_INVALID;
    }
    if (variant != FORM_CHWB && ((f->C % 8) != 0 || (f->F % 8) != 0)) { // NHWC forms move 8 channels / 8 filters at a time
        set_error("spconv_init: C and F must be multiples of 8 (got %d, %d)", f->C, f->F);
        return SHFLBW_ERR_SHAPE;
    }
    if (((uintptr_t)IFMap | (uintptr_t)OFMap) & 15) {
        set_error("spconv_init: IFMap and OFMap must be 16-byte aligned");
        return SHFLBW_ERR_INVALID;
    }
    const int Ho = (H + 2 * (f->R / 2) - f->R) / stride + 1;
    const int Wo = (W + 2 * (f->S / 2) - f->S) / stride + 1;
    if (Ho <= 0 || Wo <= 0) {
        set_error("spconv_init: empty output (%d x %d)", Ho, Wo);
        return SHFLBW_ERR_SHAPE;
    }
    if (variant < 0 || variant >= FORM_COUNT) {
        set_error("spconv_init: variant %d does not exist (0 = plane form, 1 = direct kernel, 2 = batch-innermost plane "
                  "form, 3 = batch-innermost plane form fused into one launch, 5 = patch form)", variant);
        return SHFLBW_ERR_INVALID;
    }
    if (variant == FORM_DIRECT) {
        const SpconvVariant* v = find_spconv_variant(f->brow, 0, nullptr);
        if (!v) {
            set_error("spconv_init: the direct kernel (variant 1) exists for block sizes 16, 32, 64 and 128, not %d; "
                      "the plane forms (0, 2, 3) serve every block size", f->brow);
            return SHFLBW_ERR_UNSUPPORTED;
        }
        if ((unsigned long long)B * H * W * f->C > 0x7fffffffull) {
            set_error("spconv_init: input of %d x %d x %d x %d values exceeds the 2^31 the direct kernel can index", B, H, W, f->C);
            return SHFLBW_ERR_UNSUPPORTED;
        }
        SHFLBW_HIP_TRY(v->prepare());
    }
    shflbw_device_ref ref;
    shflbw_weight_device_ref(f, &ref);
    state->args.B = B;
    state->args.H = H;
    state->args.W = W;
    state->args.C = f->C;
    state->args.F = f->F;
    state->args.R = f->R;
    state->args.S = f->S;
    state->args.stride = stride;
    state->args.A_values = ref.csb_values;
    state->args.IFMap = IFMap;
    state->args.OFMap = OFMap;
    state->args.A_bsr_indptr = ref.csb_indptr;
    state->args.A_bsr_indices = ref.csb_indices;
    state->args.A_row_indices = ref.row_permute_ids;
    state->args.alpha = 1.f; // spconv/blockwise_op.h:89-94
    state->args.beta = 0.f;
    state->Ho = Ho;
    state->Wo = Wo;
    state->packed_values = f->d_packed_values;
    state->packed_indices = (const int*)f->d_packed_indices;
    state->panel_ptr = (const int*)f->d_group_ptr;
    state->brow = f->brow;
    state->variant = variant;
    return SHFLBW_OK;
}

size_t up256(size_t n) { return (n + 255) / 256 * 256; }

// The gather ids of one (form, geometry) on the device: `ids_bytes` of slot-ordered ids, then the same ids in the
// producer-major order of every 64-slot group.  `offset_of(k)` maps a kept column k = (r*S + t)*C + c to its element
// offset in the layout-transformed input; padding slots (k < 0) get `zero_id`, the offset of a row of zeros.  Built
// and uploaded on the first call for a key, found afterwards.  The caller holds the weight's scratch_lock.
template <class OffsetOf>
int conv_ids_for(shflbw_weight* fw, const int (&key)[5], int zero_id, OffsetOf offset_of, const int** ids, const int** ids_pm)
{
    const size_t slots = fw->packed_indices.size();
    const size_t ids_bytes = up256(slots * sizeof(int) + 64);
    for (auto& e : fw->conv_ids)
        if (memcmp(e.key, key, sizeof(key)) == 0 && e.bytes == 2 * ids_bytes) {
            *ids = (const int*)e.ptr;
            *ids_pm = (const int*)((const char*)e.ptr + ids_bytes);
            return SHFLBW_OK;
        }
    std::vector<int> h(2 * ids_bytes / sizeof(int), 0);
    int* pm = h.data() + ids_bytes / sizeof(int);
    for (size_t q = 0; q < slots; q++) {
        const int k = fw->packed_indices[q];
        const int id = k < 0 ? zero_id : offset_of(k);
        h[q] = id;
        const size_t grp = q / 64; // producer-major order inside every 64-slot group
        const int j = (int)(q % 64) / 16, p = (int)(q % 16) / 4, r = (int)(q % 4);
        pm[grp * 64 + 16 * p + 4 * j + r] = id;
    }
    void* d = nullptr;
    SHFLBW_HIP_TRY(hipMalloc(&d, 2 * ids_bytes));
    if (hipMemcpy(d, h.data(), 2 * ids_bytes, hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(d);
        set_error("spconv_init: cannot upload the gather ids");
        return SHFLBW_ERR_HIP;
    }
    fw->conv_ids.push_back(shflbw_weight::ConvIds{{key[0], key[1], key[2], key[3], key[4]}, d, 2 * ids_bytes});
    *ids = (const int*)d;
    *ids_pm = (const int*)((const char*)d + ids_bytes);
    return SHFLBW_OK;
}

// The bulk scratch (layout-transformed input, filter-major result, counters) of a state: the buffer of an equal
// (form, geometry, tensors) if there is one; else a new one, cleared, while fewer than CONV_BULK_DEPTH exist; else the
// least recently handed out one - as it is when it served the same geometry (what has to be zero in it still is: the
// parts of the planes no launch writes, the counters every launch leaves at zero), freed and allocated anew
// otherwise.  The caller holds the weight's scratch_lock.
int conv_bulk_for(shflbw_weight* fw, const int (&key)[5], const void* in, const void* out, size_t bytes, char** ptr)
{
    auto& pool = fw->conv_bulk;
    fw->bulk_clock++;
    for (auto& e : pool)
        if (e.bytes == bytes && memcmp(e.key, key, sizeof(key)) == 0 && e.in == in && e.out == out) {
            e.stamp = fw->bulk_clock;
            *ptr = (char*)e.ptr;
            return SHFLBW_OK;
        }
    if ((int)pool.size() >= shflbw_weight::CONV_BULK_DEPTH) {
        size_t lru = 0;
        for (size_t i = 1; i < pool.size(); i++)
            if (pool[i].stamp < pool[lru].stamp) lru = i;
        if (pool[lru].bytes == bytes && memcmp(pool[lru].key, key, sizeof(key)) == 0) {
            pool[lru].in = in, pool[lru].out = out, pool[lru].stamp = fw->bulk_clock;
            *ptr = (char*)pool[lru].ptr;
            return SHFLBW_OK;
        }
        (void)hipFree(pool[lru].ptr);
        pool.erase(pool.begin() + lru);
    }
    void* d = nullptr;
    if (hipMalloc(&d, bytes) != hipSuccess) {
        set_error("spconv_init: cannot allocate %zu bytes of device scratch", bytes);
        return SHFLBW_ERR_HIP;
    }
    // cleared before any stream can launch on it (the caller's stream need not be ordered behind the one the clear runs on)
    if (hipMemset(d, 0, bytes) != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess) {
        (void)hipFree(d);
        set_error("spconv_init: cannot clear %zu bytes of device scratch", bytes);
        return SHFLBW_ERR_HIP;
    }
    pool.push_back(shflbw_weight::ConvBulk{{key[0], key[1], key[2], key[3], key[4]}, in, out, d, bytes, fw->bulk_clock});
    *ptr = (char*)d;
    return SHFLBW_OK;
}

// Sets up the SpMM launch in the middle of a plane form: N columns, the planes as B, `result` as D, the rewritten ids
// (element offsets: one id apart is one value apart) and `id_space` as the extent the ids address, below 2^31 values
// (every caller's size check).  `variant`: of the SpMM's variants, -1 for the library's choice among those that gather rows by id.
int bind_middle(shflbw_spconv_state* state, const shflbw_weight* f, long N, const void* planes, void* result,
                const int* ids, const int* ids_pm, long id_space, int variant = -1)
{
    int rc = spmm_init_impl(&state->spmm, f, (int)N, planes, nullptr, result, 1.f, 0.f, variant, true);
    if (rc != SHFLBW_OK) return rc;
    state->spmm.packed_indices = ids;
    state->spmm.packed_indices_pm = ids_pm;
    state->spmm.ldb_bytes = 2;
    state->spmm.args.K = (int)id_space;
    return SHFLBW_OK;
}

void copy_middle_launch_figures(shflbw_spconv_state* state)
{
    state->shared_mem_size = state->spmm.shared_mem_size;
    state->grid_dim[0] = state->spmm.grid_dim[0];
    state->block_dim[0] = state->spmm.block_dim[0];
    state->grid_dim[1] = state->grid_dim[2] = 1;
    state->block_dim[1] = state->block_dim[2] = 1;
}

// Form 0.  Points a state at its scratch (laid out by `g`) and sets up the SpMM launch in the middle.
int bind_plane_form(shflbw_spconv_state* state, const shflbw_weight* f, const PlaneForm& g, char* planes, char* result,
                    const int* ids, const int* ids_pm)
{
    state->planes = planes;
    state->result_fm = result;
    state->np = (int)g.np;
    state->plane_rows = g.PH;
    state->plane_cols = g.PW;
    state->plane_pitch = (int)g.pitch;
    state->plane_copies = g.copies;
    state->ncols = (int)g.np;
    int rc = bind_middle(state, f, g.np, planes, result, ids, ids_pm, (g.rows + 1) * g.pitch);
    if (rc != SHFLBW_OK) return rc;
    copy_middle_launch_figures(state);
    state->init_success = 1;
    return SHFLBW_OK;
}

int init_planes(shflbw_spconv_state* state, const shflbw_weight* f, int B, int H, int W, int stride, const void* IFMap,
                void* OFMap)
{
    int rc = spconv_fill_state(state, f, B, H, W, stride, IFMap, OFMap, FORM_PLANES);
    if (rc != SHFLBW_OK) return rc;
    PlaneForm g;
    if ((rc = plane_form_geometry(f, B, H, W, stride, &g)) != SHFLBW_OK) return rc;
    // The scratch cache is bookkeeping of the handle, not part of the weight's value; it is the one member an
    // init call changes, under its lock.
    shflbw_weight* fw = const_cast<shflbw_weight*>(f);
    std::lock_guard<std::mutex> scratch_guard(fw->scratch_lock);
    const int key[5] = {FORM_PLANES, B, H, W, stride};
    const int s = stride, copies = g.copies, C = f->C, S = f->S;
    const long PW = g.PW, pitch = g.pitch;
    const int *ids = nullptr, *ids_pm = nullptr;
    // kept-column id k = (r*S + t)*C + c  ->  element offset of (copy, phase, channel) row + tap offset
    rc = conv_ids_for(fw, key, (int)(g.rows * pitch), [&](int k) {
        const int c = k % C, tap = k / C, r = tap / S, t = tap % S;
        const long shift = (long)(r / s) * PW + t / s;
        const int copy = copies == 2 ? (int)(shift & 1) : 0;
        const int phase = (r % s) * s + t % s;
        return (int)((((long)copy * s * s + phase) * C + c) * pitch + shift - copy);
    }, &ids, &ids_pm);
    if (rc != SHFLBW_OK) return rc;
    char* bulk = nullptr;
    if ((rc = conv_bulk_for(fw, key, IFMap, OFMap, g.planes_bytes + g.dm_bytes, &bulk)) != SHFLBW_OK) return rc;
    return bind_plane_form(state, f, g, bulk, bulk + g.planes_bytes, ids, ids_pm);
}

// XCDs of the current device when it deals the workgroups of a launch to them the way the fused form counts on:
// consecutive workgroup ids go to consecutive XCDs, round-robin from whichever XCD the launch starts on, so a launch of
// a multiple of n workgroups puts the same number on every XCD; and every XCD has the same number of compute units.
// Checked once per device with probe launches of two sizes; 0 when the device deals differently (the fused form is
// then not offered; `why` says what was seen).
int device_xcds(std::string* why)
{
    static std::mutex lock;
    static int cached[64] = {}; // 0 = unknown, -1 = not usable
    static std::string seen[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    std::lock_guard<std::mutex> guard(lock);
    if (cached[dev] == 0) {
        cached[dev] = -1;
        const int sizes[2] = {1024, 256};
        int* d = nullptr;
        int n_all = 0;
        bool ok = hipMalloc((void**)&d, 1024 * sizeof(int)) == hipSuccess;
        if (!ok) seen[dev] = "probe allocation failed";
        for (int round = 0; ok && round < 2; round++) {
            const int blocks = sizes[round];
            std::vector<int> h(blocks, -1);
            ok = hipMemset(d, 0xff, blocks * sizeof(int)) == hipSuccess && launch_xcd_probe(d, blocks, nullptr) == hipSuccess &&
                 hipMemcpy(h.data(), d, blocks * sizeof(int), hipMemcpyDeviceToHost) == hipSuccess;
            if (!ok) {
                seen[dev] = "probe launch failed";
                break;
            }
            int n = 0;
            for (int v : h) n = std::max(n, v + 1);
            ok = n >= 1 && n <= 8 && (round == 0 || n == n_all) && device_compute_units() % n == 0 && h[0] >= 0;
            for (int i = 0; ok && i < blocks; i++) ok = h[i] == (h[0] + i) % n;
            n_all = n;
            if (!ok) {
                char buf[256];
                int len = snprintf(buf, sizeof(buf), "launch of %d workgroups, %d XCD ids, workgroups 0.. ran on XCDs", blocks, n);
                for (int i = 0; i < 24 && len < (int)sizeof(buf) - 8; i++) len += snprintf(buf + len, sizeof(buf) - len, " %d", h[i]);
                seen[dev] = buf;
            }
        }
        if (d) (void)hipFree(d);
        if (ok) cached[dev] = n_all;
    }
    if (why) *why = seen[dev];
    return cached[dev] > 0 ? cached[dev] : 0;
}

// Geometry of the batch-innermost plane forms (2, 3, 4): phase planes planes[phase (a, b)][c][(i * PW + j) * B + img] =
// in(i * stride + a - R/2, j * stride + b - S/2) of image img and channel c, PHX = Ho + (R-1)/stride rows and
// PW = Wo + (S-1)/stride columns.  Every tap offset is a multiple of B values, 16 bytes or more: one copy of the planes
// serves all taps.  The GEMM runs over the Ho * PW * B columns (ho, j, img) of the padded output grid.
struct BatchPlanes {
    int Ho, Wo;
    long PHX, PW;
    long np;        // values of one channel plane
    long rows;      // channel rows: stride^2 * C
    long ncols;     // columns of the GEMM
    long max_shift; // largest tap offset in values
};

void batch_planes_geometry(const shflbw_weight* f, int B, int stride, int Ho, int Wo, BatchPlanes* g)
{
    const int s = stride;
    g->Ho = Ho, g->Wo = Wo;
    g->PHX = Ho + (f->R - 1) / s;
    g->PW = Wo + (f->S - 1) / s;
    g->np = g->PHX * g->PW * B;
    g->rows = (long)s * s * f->C;
    g->ncols = (long)Ho * g->PW * B;
    g->max_shift = ((long)((f->R - 1) / s) * g->PW + (f->S - 1) / s) * B;
}

// Strides past the map read it at the first row and column only, whatever they are: one such stride stands for all.
long chwb_stride(int H, int W, int R, int S, int stride) { return std::min((long)stride, (long)H + W + R + S); }

// Form 4 over the input itself (the state holds no planes): where the ids of its taps fit (chwb_tap_id), the output does
// not overwrite what is still to be gathered, and the input row of every position times the width of the filter stays
// within an int (by which the kernel tells the taps outside the map).
bool chwb_gathers_input(const shflbw_weight* f, int B, int H, int W, int stride, const void* IFMap, const void* OFMap)
{
    const size_t pixels = (size_t)B * H * W * 2;
    const char *in = (const char*)IFMap, *out = (const char*)OFMap;
    const bool apart = in + pixels * f->C <= out || out + pixels * f->F <= in;
    return apart && (long)f->R * f->S <= CHWB_MAX_TAPS &&
           ((unsigned long long)f->C * H * W + (unsigned long long)f->R * W + f->S) * (unsigned long long)B * 2ull < 0x80000000ull &&
           std::max(H, W) * chwb_stride(H, W, f->R, f->S, stride) * f->S < 0x7fffffffL;
}

int init_chwb_taps(shflbw_spconv_state* state, const shflbw_weight* f, int B, int H, int W, int stride, const void* IFMap, void* OFMap)
{
    const long ncols = (long)H * W * B; // columns of the GEMM: the output positions (ho, wo, b)
    if (ncols > 0x7fffffffL) {
        set_error("spconv_init: problem too large (%ld output positions)", ncols);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    // The cut of the SpMM of these sizes.  With three widths by the number of tiles, and one width for block height 16, us, before / now:
    // 16 x 14 x 14 x 656 -> 32, 3 x 3, block height 16 20.4 / 11.9, 8 x 7 x 7 x 304 -> 1152, 5 x 5, 14.3 / 11.0; block height 32, 32 x 55 x 27 x
    // 360 -> 128, 1 x 7, 20.1 / 18.5.  The estimate was fitted to no convolution; over 500 drawn layers, every cut timed, its choice takes
    // 1.013 times the fastest cut's time, 1.24 at worst.
    const int variant = auto_spmm_variant(f, (int)ncols, false, false, device_compute_units());
    const SpmmVariant* v = find_spmm_variant(f->brow, variant, nullptr);
    const ConvTapsKernel* k = v ? conv_taps_kernel(v->name) : nullptr;
    if (!k) {
        set_error("spconv_init: no kernel for block size %d", f->brow);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    SHFLBW_HIP_TRY(k->prepare());
    state->middle_tile_cols = v->BN;
    shflbw_weight* fw = const_cast<shflbw_weight*>(f); // the table of ids is bookkeeping of the handle (see init_planes)
    std::lock_guard<std::mutex> scratch_guard(fw->scratch_lock);
    const int key[5] = {FORM_CHWB, B, H, W, 0}; // the same for every stride
    const int C = f->C, S = f->S;
    const int *ids = nullptr, *ids_pm = nullptr;
    int rc = conv_ids_for(fw, key, chwb_tap_id(0, CHWB_MAX_TAPS), [&](int kk) {
        const int c = kk % C, tap = kk / C, r = tap / S, t = tap % S;
        return chwb_tap_id((unsigned)((((long)c * H + r) * W + t) * (B / 8)), (unsigned)tap);
    }, &ids, &ids_pm);
    if (rc != SHFLBW_OK) return rc;
    state->ncols = (int)ncols;
    if ((rc = bind_middle(state, f, ncols, IFMap, OFMap, ids, ids_pm, (long)C * H * W * B, variant)) != SHFLBW_OK) return rc;
    state->shared_mem_size = (size_t)v->lds_bytes;
    state->grid_dim[0] = (unsigned)((f->nrow / f->brow) * ((ncols + v->BN - 1) / v->BN));
    state->block_dim[0] = (unsigned)v->threads;
    state->grid_dim[1] = state->grid_dim[2] = 1;
    state->block_dim[1] = state->block_dim[2] = 1;
    state->init_success = 1;
    return SHFLBW_OK;
}

//   form 4: the caller's tensors are C-H-W-B / F-H-W-B (the reference's), H and W bound input and output alike,
//           the SpMM writes OFMap itself (its epilogue drops the padding columns, output_column()); only for what
//           chwb_gathers_input() leaves;
//   form 2: the caller's tensors are NHWC with true stride and padding; the SpMM writes result_fm[f][(ho, wo, img)],
//           a tile transpose writes OFMap.
int init_batch_planes(shflbw_spconv_state* state, const shflbw_weight* f, int B, int H, int W, int stride,
                      const void* IFMap, void* OFMap, int variant)
{
    int rc = spconv_fill_state(state, f, B, H, W, stride, IFMap, OFMap, variant);
    if (rc != SHFLBW_OK) return rc;
    if (B % 8 != 0) { // the reference's kernel moves 8 batch entries at a time too (spconv/blockwise_kernel.h:200-207)
        set_error("spconv_init: the batch must be a multiple of 8 for this form (got %d)", B);
        return SHFLBW_ERR_SHAPE;
    }
    if (variant == FORM_CHWB) { // H and W are the extents of the output grid and the bounds of the input (spconv/blockwise_format.h:111-115)
        state->Ho = H;
        state->Wo = W;
        if (chwb_gathers_input(f, B, H, W, stride, IFMap, OFMap)) return init_chwb_taps(state, f, B, H, W, stride, IFMap, OFMap);
    }
    if (stride > 5792) { // stride^2 planes of 64 values or more: beyond 4 GiB
        set_error("spconv_init: stride %d has too many phase planes", stride);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    BatchPlanes g;
    batch_planes_geometry(f, B, stride, state->Ho, state->Wo, &g);
    // the SpMM in the middle: tile width by the size of the GEMM, as for the SpMM proper
    const ConvChwbKernel* k = conv_chwb_kernel(f->brow, 0, f->nrow / f->brow, g.ncols, device_compute_units());
    if (!k) {
        set_error("spconv_init: no kernel for block size %d", f->brow);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    SHFLBW_HIP_TRY(k->prepare());
    state->middle_tile_cols = k->BN;
    const int s = stride, C = f->C, S = f->S;
    const long pitch = (g.np + g.max_shift + 8 + 63) / 64 * 64;
    if (g.ncols > 0x7fffffffL || !planes_fit(g.rows, pitch)) {
        set_error("spconv_init: problem too large (%ld channel rows of %ld values)", g.rows, pitch);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    const size_t planes_bytes = up256((size_t)(g.rows + 1) * pitch * 2); // one more row: zeros, for the padding slots
    const size_t dm_bytes = variant == FORM_BPLANES ? up256((size_t)f->F * g.Ho * g.Wo * B * 2) : 0;
    shflbw_weight* fw = const_cast<shflbw_weight*>(f); // the scratch cache is bookkeeping of the handle (see init_planes)
    std::lock_guard<std::mutex> scratch_guard(fw->scratch_lock);
    const int key[5] = {variant, B, H, W, stride};
    const long PW = g.PW;
    const int *ids = nullptr, *ids_pm = nullptr;
    // kept-column id k = (r*S + t)*C + c  ->  element offset of the (phase, channel) row + tap offset
    rc = conv_ids_for(fw, key, (int)(g.rows * pitch), [&](int kk) {
        const int c = kk % C, tap = kk / C, r = tap / S, t = tap % S;
        return (int)((((long)(r % s) * s + t % s) * C + c) * pitch + ((long)(r / s) * PW + t / s) * B);
    }, &ids, &ids_pm);
    if (rc != SHFLBW_OK) return rc;
    char* bulk = nullptr;
    if ((rc = conv_bulk_for(fw, key, IFMap, OFMap, planes_bytes + dm_bytes, &bulk)) != SHFLBW_OK) return rc;
    state->planes = bulk;
    state->result_fm = variant == FORM_BPLANES ? bulk + planes_bytes : nullptr;
    state->np = (int)g.np;
    state->plane_rows = (int)g.PHX;
    state->plane_cols = (int)g.PW;
    state->plane_pitch = (int)pitch;
    state->plane_copies = 1;
    state->ncols = (int)g.ncols;
    // the SpMM in the middle: row f of its result is the row of filter f, in OFMap itself (form 4) or in result_fm
    rc = bind_middle(state, f, g.ncols, state->planes, variant == FORM_BPLANES ? state->result_fm : OFMap, ids, ids_pm,
                     (g.rows + 1) * pitch);
    if (rc != SHFLBW_OK) return rc;
    state->shared_mem_size = (size_t)k->lds_bytes;
    state->grid_dim[0] = (unsigned)((f->nrow / f->brow) * ((g.ncols + k->BN - 1) / k->BN));
    state->block_dim[0] = (unsigned)k->threads;
    state->grid_dim[1] = state->grid_dim[2] = 1;
    state->block_dim[1] = state->block_dim[2] = 1;
    state->init_success = 1;
    return SHFLBW_OK;
}

// Layout of the fused form's bulk scratch: nx slabs of planes | nx filter-major results | counters.
struct FusedForm {
    BatchPlanes g;
    int nx;          // XCDs of the device
    long cx;         // columns of the GEMM per XCD (a multiple of 64)
    long pitch;      // values per channel row of a slab: cx + the largest tap offset, rounded up to 64
    size_t slab_bytes, fm_bytes, sync_bytes;
    size_t total_bytes() const { return (size_t)nx * (slab_bytes + fm_bytes) + sync_bytes; }
};

int fused_form_geometry(const shflbw_weight* f, int B, int stride, int Ho, int Wo, int nx, FusedForm* g)
{
    if (stride > 5) {
        set_error("spconv_init: stride %d has too many phase planes for the fused form", stride);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    batch_planes_geometry(f, B, stride, Ho, Wo, &g->g);
    g->nx = nx;
    g->cx = ((g->g.ncols + nx - 1) / nx + 63) / 64 * 64;
    g->pitch = (g->cx + g->g.max_shift + 63) / 64 * 64;
    if (g->g.ncols > 0x7fffffffL ||
        (unsigned long long)(g->g.rows + 1) * (unsigned long long)g->pitch * 2ull > 0x7fffffffull ||
        (unsigned long long)f->F * (unsigned long long)g->cx > 0x7fffffffull) {
        set_error("spconv_init: problem too large for the fused form (%ld channel rows of %ld values per XCD)", g->g.rows, g->pitch);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    g->slab_bytes = up256((size_t)(g->g.rows + 1) * g->pitch * 2); // one more row: zeros, for the padding slots
    g->fm_bytes = up256((size_t)f->F * g->cx * 2);
    g->sync_bytes = (size_t)conv_xcd_sync_lines(nx) * SYNC_LINE * sizeof(int);
    return SHFLBW_OK;
}

// form 3: NHWC tensors, the three steps of form 2 in one launch, every XCD on its own columns (spconv_xcd_kernel)
int init_fused(shflbw_spconv_state* state, const shflbw_weight* f, int B, int H, int W, int stride, const void* IFMap,
               void* OFMap)
{
    int rc = spconv_fill_state(state, f, B, H, W, stride, IFMap, OFMap, FORM_FUSED);
    if (rc != SHFLBW_OK) return rc;
    if (B % 8 != 0) {
        set_error("spconv_init: the batch must be a multiple of 8 for this form (got %d)", B);
        return SHFLBW_ERR_SHAPE;
    }
    const ConvXcdKernel* k = conv_xcd_kernel(f->brow);
    if (!k) {
        set_error("spconv_init: no fused kernel for block size %d", f->brow);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    std::string why;
    const int nx = device_xcds(&why);
    if (nx <= 0) {
        set_error("spconv_init: this device does not deal workgroups to its XCDs in the way the fused form counts on (%s)", why.c_str());
        return SHFLBW_ERR_UNSUPPORTED;
    }
    if (device_compute_units() / nx > 32) {
        set_error("spconv_init: the fused form numbers at most 32 workgroups per XCD (this device: %d)", device_compute_units() / nx);
        return SHFLBW_ERR_UNSUPPORTED;
    }
    SHFLBW_HIP_TRY(k->prepare());
    FusedForm g;
    if ((rc = fused_form_geometry(f, B, stride, state->Ho, state->Wo, nx, &g)) != SHFLBW_OK) return rc;
    const int s = stride, C = f->C, S = f->S;
    const long PW = g.g.PW, pitch = g.pitch;
    shflbw_weight* fw = const_cast<shflbw_weight*>(f); // the scratch cache is bookkeeping of the handle (see init_planes)
    std::lock_guard<std::mutex> scratch_guard(fw->scratch_lock);
    const int key[5] = {FORM_FUSED, B, H, W, stride};
    const int *ids = nullptr, *ids_pm = nullptr;
    // kept-column id k = (r*S + t)*C + c  ->  element offset inside a slab: (phase, channel) row + tap offset
    rc = conv_ids_for(fw, key, (int)(g.g.rows * pitch), [&](int kk) {
        const int c = kk % C, tap = kk / C, r = tap / S, t = tap % S;
        return (int)((((long)(r % s) * s + t % s) * C + c) * pitch + ((long)(r / s) * PW + t / s) * B);
    }, &ids, &ids_pm);
    if (rc != SHFLBW_OK) return rc;
    char* bulk = nullptr;
    if ((rc = conv_bulk_for(fw, key, IFMap, OFMap, g.total_bytes(), &bulk)) != SHFLBW_OK) return rc;
    state->planes = bulk;
    state->result_fm = bulk + (size_t)nx * g.slab_bytes;
    state->sync = bulk + (size_t)nx * (g.slab_bytes + g.fm_bytes);
    state->np = (int)g.g.np;
    state->plane_rows = (int)g.g.PHX;
    state->plane_cols = (int)g.g.PW;
    state->plane_pitch = (int)pitch;
    state->plane_copies = 1;
    state->ncols = (int)g.g.ncols;
    state->xcds = nx;
    state->cols_per_xcd = (int)g.cx;
    state->patience_ticks = 5000; // 50 us
    // the SpMM in the middle, as one XCD sees it: cx columns, its slab as B, its result as D
    rc = bind_middle(state, f, g.cx, state->planes, state->result_fm, ids, ids_pm, (g.g.rows + 1) * pitch);
    if (rc != SHFLBW_OK) return rc;
    state->shared_mem_size = (size_t)k->lds_bytes;
    state->grid_dim[0] = (unsigned)(device_compute_units() / nx * nx);
    state->block_dim[0] = (unsigned)k->threads;
    state->grid_dim[1] = state->grid_dim[2] = 1;
    state->block_dim[1] = state->block_dim[2] = 1;
    state->init_success = 1;
    return SHFLBW_OK;
}

// The filters of every workgroup of `rows_wg` rows in output order, and the place of each row among them.
void fill_patch_places(const shflbw_weight* fw, int rows_wg, int* filt, unsigned short* dst)
{
    const int F = fw->F;
    std::vector<int> row_of(F), next((F + rows_wg - 1) / rows_wg, 0);
    for (int i = 0; i < F; i++) row_of[fw->row_permute ? fw->row_permute_ids[i] : i] = i;
    for (int filter = 0; filter < F; filter++) {
        const int chunk = row_of[filter] / rows_wg, place = next[chunk]++;
        filt[chunk * rows_wg + place] = filter;
        dst[row_of[filter]] = (unsigned short)place;
    }
}

const shflbw_weight::PatchPlaces* find_patch_places(const shflbw_weight* fw, int rows_wg)
{
    for (auto& e : fw->patch_places)
        if (e.rows_wg == rows_wg) return &e;
    return nullptr;
}

// The places of a cut: found, or built and uploaded.  The caller holds the weight's scratch_lock.
int patch_places_for(shflbw_weight* fw, int rows_wg, const shflbw_weight::PatchPlaces** out)
{
    if ((*out = find_patch_places(fw, rows_wg))) return SHFLBW_OK;
    shflbw_weight::PatchPlaces e{rows_wg, nullptr, 0, nullptr, nullptr};
    const size_t o_dst = up256((size_t)fw->F * sizeof(int));
    e.bytes = o_dst + up256((size_t)fw->F * sizeof(unsigned short));
    std::vector<unsigned char> h(e.bytes, 0);
    fill_patch_places(fw, rows_wg, (int*)h.data(), (unsigned short*)(h.data() + o_dst));
    SHFLBW_HIP_TRY(hipMalloc(&e.ptr, e.bytes));
    if (hipMemcpy(e.ptr, h.data(), e.bytes, hipMemcpyHostToDevice) != hipSuccess) {
        (void)hipFree(e.ptr);
        set_error("spconv_init: cannot upload the output places of the patch form");
        return SHFLBW_ERR_HIP;
    }
    e.filt = (const int*)e.ptr;
    e.dst = (const unsigned short*)((const char*)e.ptr + o_dst);
    fw->patch_places.push_back(e);
    *out = &fw->patch_places.back();
    return SHFLBW_OK;
}

// The filter as the patch form reads it, for patches of the shape of `p`: built on the first call for a shape, found
// afterwards; null in *out where CONV_PATCH_IMAGES others are held.  With it go the places of that cut, one copy for both.  The
// caller holds the weight's scratch_lock.
int patch_image_for(shflbw_weight* fw, const ConvPatchPlan& p, const shflbw_weight::PatchImage** out)
{
    *out = nullptr;
    const int V = fw->brow, X = fw->nrow / V, F = fw->F, C = fw->C, S = fw->S;
    const int RW = conv_patch_unit_rows(V), per_panel = V / RW, nunits = F / RW;
    const ConvPatchShape shape = conv_patch_shape(RW, p);
    for (auto& e : fw->patch_images)
        if (e.shape == shape) {
            *out = &e;
            return SHFLBW_OK;
        }
    if ((int)fw->patch_images.size() >= shflbw_weight::CONV_PATCH_IMAGES) return SHFLBW_OK;
    shflbw_weight::PatchImage e{};
    e.shape = shape;
    size_t batches = 0;
    for (int i = 0; i < X; i++) batches += (size_t)((fw->indptr[i + 1] - fw->indptr[i] + 31) / 32) * per_panel;
    const size_t held = batches + CONV_PATCH_TAIL_BATCHES;
    const size_t o_offs = up256(held * 32 * RW * sizeof(uint16_t)), o_first = o_offs + up256(held * 32 * sizeof(uint16_t));
    const size_t o_filt = o_first + up256((size_t)(nunits + 1) * sizeof(int)), o_dst = o_filt + up256((size_t)F * sizeof(int));
    const size_t o_src = o_dst + up256((size_t)F * sizeof(unsigned short));
    e.bytes = o_src + up256(batches * 32 * sizeof(int));
    e.touch = o_filt;
    // The fragments, many times the size of the tables, are packed on the device from the weight's values once packing and
    // copying them costs more than a launch and a wait (first initialisation of a filter, fragments packed on the host / on
    // the device: 72 KB 29 / 43 us, 144 KB 38 / 48, 288 KB 59 / 58 and 47 / 47, 576 KB 79 / 59, 1843 KB 329 / 211).
    const bool on_host = o_offs <= 256u << 10;
    const size_t o_host = on_host ? 0 : o_offs; // what is made here starts there
    std::vector<unsigned char> h(e.bytes - o_host, 0);
    uint16_t* A = (uint16_t*)h.data(); // on_host
    uint16_t* offs = (uint16_t*)(h.data() + (o_offs - o_host));
    int* first = (int*)(h.data() + (o_first - o_host));
    int* src = (int*)(h.data() + (o_src - o_host));
    // slots of the groups a batch's reads are made of, group after group: a pass reads slots 8 (lane / 16 or
    // lane / 32) + 0..3 of a step, the second read of a fragment the four behind them.  A lane addresses slots s and
    // s + 4 of a step and loads the offsets of all steps of a batch at once.
    int slot_of[32], place_of[32];
    for (int t = 0; t < 32; t++) {
        const int s = RW == 16 ? (t / 16) * 16 + ((t / 8) & 1) * 4 + ((t / 4) & 1) * 8 + t % 4 : t;
        const int in_step = RW == 16 ? s : s % 16, step = RW == 16 ? 0 : s / 16;
        const int pair = (in_step / 8) * 4 + in_step % 4, hi = (in_step % 8) / 4;
        slot_of[t] = s;
        place_of[t] = RW == 16 ? pair * 2 + hi : pair * 4 + step * 2 + hi;
    }
    // LDS offset (in 8 bytes) of every column, tap after tap
    std::vector<uint16_t> at(fw->ncol);
    for (int r = 0, k = 0; r < fw->R; r++)
        for (int t = 0; t < S; t++)
            for (int c = 0; c < C; c++, k++) at[k] = (uint16_t)((c * p.pitch >> 3) + r * p.patch_w + t);
    const uint16_t zero_row = (uint16_t)(C * p.pitch >> 3);
    const ConvPatchOrder keep_apart(shape.foot, conv_patch_group(RW));
    std::vector<int> pair_of, order;
    static const uint16_t zeros[64] = {};
    size_t b = 0;
    for (int panel = 0; panel < X; panel++) {
        const int begin = fw->indptr[panel], nnz = fw->indptr[panel + 1] - begin;
        pair_of.resize(nnz);
        for (int i = 0; i < nnz; i++) pair_of[i] = at[fw->indices[begin + i]] & 31;
        keep_apart.of(pair_of, order);
        for (int part = 0; part < per_panel; part++) {
            first[panel * per_panel + part] = (int)b;
            for (int t0 = 0; t0 < nnz; t0 += 32) {
                uint16_t* o = offs + (b + t0 / 32) * 32;
                int* from = src + (b + t0 / 32) * 32;
                for (int t = 0; t < 32; t++) {
                    const bool held = t0 + t < nnz;
                    const int i = begin + (held ? order[t0 + t] : 0);
                    o[place_of[t]] = held ? at[fw->indices[i]] : zero_row;
                    from[slot_of[t]] = held ? i * per_panel + part : -1;
                }
                for (int s = 0; on_host && s < 32; s += 8) {
                    const uint16_t* v[8];
                    for (int j = 0; j < 8; j++) v[j] = from[s + j] < 0 ? zeros : fw->values.data() + (size_t)from[s + j] * RW;
                    uint16_t* a = A + (b + t0 / 32) * 32 * RW;
                    if (RW == 16) {
                        interleave8(v, 16, a + (s / 8) * 16 * 8);
                        continue;
                    }
                    for (int mb = 0; mb < RW / 32; mb++) {
                        interleave8(v, 32, a + ((size_t)((s / 16) * (RW / 32) + mb) * 64 + (s % 16) / 8 * 32) * 8);
                        for (int j = 0; j < 8; j++) v[j] += 32;
                    }
                }
            }
            b += (nnz + 31) / 32;
        }
    }
    first[nunits] = (int)b;
    const bool with_places = !find_patch_places(fw, p.rows_wg);
    if (with_places) fill_patch_places(fw, p.rows_wg, (int*)(h.data() + (o_filt - o_host)), (unsigned short*)(h.data() + (o_dst - o_host)));
    SHFLBW_HIP_TRY(hipMalloc(&e.ptr, e.bytes));
    hipError_t err = hipMemcpy((char*)e.ptr + o_host, h.data(), h.size(), hipMemcpyHostToDevice);
    if (err == hipSuccess && !on_host) {
        err = launch_patch_pack((const half_t*)fw->d_values, (const int*)((char*)e.ptr + o_src), (half8_t*)e.ptr, RW, batches, nullptr);
        if (err == hipSuccess) err = hipStreamSynchronize(nullptr); // any stream may launch on the image
    }
    if (err != hipSuccess) {
        (void)hipFree(e.ptr);
        set_error("spconv_init: cannot build the filter image of the patch form: %s", hipGetErrorString(err));
        return SHFLBW_ERR_HIP;
    }
    e.offs = (const unsigned short*)((const char*)e.ptr + o_offs);
    e.first_batch = (const int*)((const char*)e.ptr + o_first);
    fw->patch_images.push_back(e);
    if (with_places)
        fw->patch_places.push_back({p.rows_wg, nullptr, 0, (const int*)((const char*)e.ptr + o_filt), (const unsigned short*)((const char*)e.ptr + o_dst)});
    *out = &fw->patch_images.back();
    return SHFLBW_OK;
}

// The cut of one geometry of a filter and its launch arguments, as a copy.  SHFLBW_ERR_UNSUPPORTED when no patch fits or,
// unless `forced`, the plane forms are estimated faster; SHFLBW_ERR_CAPACITY when that is so only because the filter's images
// are all taken by other shapes.
int conv_patch_for(shflbw_weight* fw, int B, int H, int W, int stride, int Ho, int Wo, bool forced, ConvPatchArgs* out)
{
    std::lock_guard<std::mutex> scratch_guard(fw->scratch_lock);
    auto& all = fw->patch_geometries;
    shflbw_weight::PatchGeometry* g = nullptr;
    for (auto& e : all)
        if (e.key[0] == B && e.key[1] == H && e.key[2] == W && e.key[3] == stride) g = &e;
    const ConvPatchProblem q{fw->brow, fw->F, fw->C, fw->R, fw->S, (double)fw->nnzb / (fw->nrow / fw->brow), fw->row_permute ? 1 : 0,
                             B, H, W, Ho, Wo, stride, device_compute_units()};
    if (!g) {
        if ((int)all.size() < shflbw_weight::CONV_PATCH_GEOMETRIES)
            g = &*all.insert(all.end(), shflbw_weight::PatchGeometry{});
        else
            g = &*std::min_element(all.begin(), all.end(), [](const auto& x, const auto& y) { return x.stamp < y.stamp; });
        *g = shflbw_weight::PatchGeometry{{B, H, W, stride}, {}, 0, {}, 0};
        conv_patch_plan(q, &g->plan);
    }
    g->stamp = ++fw->bulk_clock;
    if (!g->plan.valid || !(forced || g->plan.preferred)) return SHFLBW_ERR_UNSUPPORTED;
    if (!g->bound) {
        const int RW = conv_patch_unit_rows(fw->brow);
        ConvPatchPlan plan = g->plan;
        const shflbw_weight::PatchImage* image = nullptr;
        int rc = patch_image_for(fw, plan, &image);
        if (rc != SHFLBW_OK) return rc;
        if (!image) { // no room for another shape: the best cut among those that are held
            std::vector<ConvPatchShape> held;
            for (auto& e : fw->patch_images) held.push_back(e.shape);
            if (!conv_patch_plan(q, &plan, &held) || !(forced || plan.preferred)) return SHFLBW_ERR_CAPACITY;
            if ((rc = patch_image_for(fw, plan, &image)) != SHFLBW_OK) return rc;
        }
        const shflbw_weight::PatchPlaces* places = nullptr;
        if ((rc = patch_places_for(fw, plan.rows_wg, &places)) != SHFLBW_OK) return rc;
        SHFLBW_HIP_TRY(conv_patch_kernel(RW, plan.col_blocks, plan.waves, plan.deep)->prepare());
        // (an image beyond three quarters of an XCD's L2 is left to the ring past that)
        plan.touch_bytes = (unsigned)std::min<size_t>(image->touch, 3u << 20) - 4;
        plan.touch_step = (unsigned)(plan.jobs_per_xcd * plan.waves * 64) * 128u;
        ConvPatchArgs& a = g->args;
        a.p = plan;
        a.C = fw->C, a.F = fw->F, a.R = fw->R, a.S = fw->S;
        a.in = nullptr, a.out = nullptr, a.streams = 0; // each launch's own
        a.packedA = (const half8_t*)image->ptr;
        a.first_batch = image->first_batch;
        a.offs = image->offs;
        a.dst = places->dst;
        a.filt = places->filt;
        a.dense = !fw->row_permute || plan.chunks == 1;
        g->bound = 1;
    }
    *out = g->args;
    return SHFLBW_OK;
}

// Form 5.  `forced`: whatever the estimate says.  SHFLBW_ERR_UNSUPPORTED when the form does not take the geometry.
int init_patch(shflbw_spconv_state* state, const shflbw_weight* f, int B, int H, int W, int stride, const void* IFMap,
               void* OFMap, bool forced)
{
    int rc = spconv_fill_state(state, f, B, H, W, stride, IFMap, OFMap, FORM_PATCH);
    if (rc != SHFLBW_OK) return rc;
    ConvPatchArgs args;
    rc = conv_patch_for(const_cast<shflbw_weight*>(f), B, H, W, stride, state->Ho, state->Wo, forced, &args);
    if (rc == SHFLBW_ERR_UNSUPPORTED)
        set_error(forced ? "spconv_init: no input patch of a workgroup fits the LDS (%d channels, %d x %d filter), or the tensors leave 32-bit indexes"
                         : "spconv_init: the patch form does not take this layer (%d channels, %d x %d filter)", f->C, f->R, f->S);
    if (rc == SHFLBW_ERR_CAPACITY)
        set_error("spconv_init: the filter holds %d images of the patch form already, none of which suits this layer "
                  "(shflbw_weight_release_scratch frees them)", shflbw_weight::CONV_PATCH_IMAGES);
    if (rc != SHFLBW_OK) return rc;
    static_assert(sizeof(ConvPatchArgs) <= sizeof(state->patch_launch) && std::is_trivially_copyable<ConvPatchArgs>::value, "kept in the state");
    memcpy(state->patch_launch, &args, sizeof(args));
    state->patch = args.packedA;
    state->ncols = B * state->Ho * state->Wo;
    state->shared_mem_size = (size_t)args.p.lds_bytes;
    state->grid_dim[0] = (unsigned)args.p.jobs;
    state->block_dim[0] = (unsigned)(args.p.waves * 64);
    state->grid_dim[1] = state->grid_dim[2] = 1;
    state->block_dim[1] = state->block_dim[2] = 1;
    state->init_success = 1;
    return SHFLBW_OK;
}

// launch arguments every form shares
void fill_conv_launch_args(const shflbw_spconv_state* state, SpconvLaunchArgs* out)
{
    SpconvLaunchArgs& a = *out;
    a.B = state->args.B;
    a.H = state->args.H;
    a.W = state->args.W;
    a.C = state->args.C;
    a.F = state->args.F;
    a.R = state->args.R;
    a.S = state->args.S;
    a.stride = state->args.stride;
    a.pad_h = a.R / 2;
    a.pad_w = a.S / 2;
    a.Ho = state->Ho;
    a.Wo = state->Wo;
    a.X = a.F / state->brow;
    a.n_tiles = 0;
    a.packedA = (const half8_t*)state->packed_values;
    a.kidx = state->packed_indices;
    a.panel_desc = state->panel_ptr;
    a.row_ids = state->args.A_row_indices;
    a.in = (const half_t*)state->args.IFMap;
    a.out = (half_t*)state->args.OFMap;
}

// Chunks of the layout phases of the fused form: `tiles` = 8, 4 or 2 tiles of 64 x 64 per chunk, as many of them
// along the contiguous axis of the source (`along` tiles there) as there are.  Picks the chunk size that needs the
// fewest rounds of the `workers` workgroups of an XCD, a round costing its tiles plus a fixed latency of about
// four tiles' worth.
void pick_chunk(int along_tiles, int across_tiles, int workers, int* t_along, int* t_across, int* chunks_along)
{
    auto pow2_le = [](int n, int cap) { int p = 1; while (p * 2 <= n && p * 2 <= cap) p *= 2; return p; };
    long best_cost = -1;
    for (int tiles = 8; tiles >= 2; tiles >>= 1) {
        const int ta = pow2_le(along_tiles, tiles), tb = tiles / ta;
        const long chunks = (long)((along_tiles + ta - 1) / ta) * ((across_tiles + tb - 1) / tb);
        const long rounds = (chunks + workers - 1) / workers;
        const long cost = rounds * (tiles + 4);
        if (best_cost < 0 || cost < best_cost) {
            best_cost = cost;
            *t_along = ta, *t_across = tb, *chunks_along = (along_tiles + ta - 1) / ta;
        }
    }
}

} // namespace

extern "C" {

int shflbw_spconv_init_variant(shflbw_spconv_state* state, const shflbw_weight* f, int B, int H, int W, int stride,
                               const void* IFMap, void* OFMap, int variant)
{
    if (variant == FORM_CHWB) {
        if (state) memset(state, 0, sizeof(*state));
        set_error("spconv_init: form 4 works on C-H-W-B / F-H-W-B tensors; call shflbw_spconv_init_chwb");
        return SHFLBW_ERR_INVALID;
    }
    // the library's choice: the patch form wherever it is estimated faster; else the batch-innermost form wherever the batch
    // allows it (one copy of the planes instead of two, no dead plane rows in the result; with the tile width of its SpMM
    // chosen by the size of the GEMM it is level with the plane form on the smallest layers and ahead from a few hundred
    // output pixels on), else the plane form
    if (variant < 0) {
        const int rc = init_patch(state, f, B, H, W, stride, IFMap, OFMap, false);
        if (rc != SHFLBW_ERR_UNSUPPORTED && rc != SHFLBW_ERR_CAPACITY) return rc;
        variant = B % 8 == 0 ? FORM_BPLANES : FORM_PLANES;
    }
    if (variant == FORM_PATCH) return init_patch(state, f, B, H, W, stride, IFMap, OFMap, true);
    if (variant == FORM_BPLANES) return init_batch_planes(state, f, B, H, W, stride, IFMap, OFMap, FORM_BPLANES);
    if (variant == FORM_FUSED) return init_fused(state, f, B, H, W, stride, IFMap, OFMap);
    if (variant == FORM_PLANES) return init_planes(state, f, B, H, W, stride, IFMap, OFMap);
    int rc = spconv_fill_state(state, f, B, H, W, stride, IFMap, OFMap, variant);
    if (rc != SHFLBW_OK) return rc;
    // the direct kernel
    const SpconvVariant* v = find_spconv_variant(f->brow, 0, nullptr);
    const long npix = (long)B * state->Ho * state->Wo;
    state->shared_mem_size = (size_t)v->lds_bytes;
    state->grid_dim[0] = (unsigned)((f->F / f->brow) * ((npix + v->BN - 1) / v->BN));
    state->block_dim[0] = (unsigned)v->threads;
    state->grid_dim[1] = state->grid_dim[2] = 1;
    state->block_dim[1] = state->block_dim[2] = 1;
    state->init_success = 1;
    return SHFLBW_OK;
}

int shflbw_spconv_init_chwb(shflbw_spconv_state* state, const shflbw_weight* f, int B, int H, int W, int stride,
                            const void* IFMap, void* OFMap)
{
    return init_batch_planes(state, f, B, H, W, stride, IFMap, OFMap, FORM_CHWB);
}

int shflbw_spconv_exec(const shflbw_spconv_state* state, void* stream)
{
    if (!state || !state->init_success) {
        set_error("spconv_exec: state was not initialised successfully");
        return SHFLBW_ERR_STATE;
    }
    hipError_t e = hipSuccess;
    if (state->variant == FORM_PATCH) {
        ConvPatchArgs p;
        memcpy(&p, state->patch_launch, sizeof(p));
        const ConvPatchKernel* k = conv_patch_kernel(conv_patch_unit_rows(state->brow), p.p.col_blocks, p.p.waves, p.p.deep);
        if (!k) return SHFLBW_ERR_UNSUPPORTED;
        p.in = (const half_t*)state->args.IFMap;
        p.out = (half_t*)state->args.OFMap;
        p.streams = conv_patch_streams((size_t)state->ncols * (size_t)p.F * 2);
        e = k->launch(p, (hipStream_t)stream);
        if (e == hipSuccess) return SHFLBW_OK;
        set_error("spconv_exec: launch failed: %s", hipGetErrorString(e));
        return SHFLBW_ERR_HIP;
    }
    SpconvLaunchArgs a;
    fill_conv_launch_args(state, &a);
    if (state->variant == FORM_CHWB || state->variant == FORM_BPLANES) {
        if (!state->planes) { // form 4 over the input itself
            const SpmmVariant* v = find_spmm_variant(state->brow, state->spmm.variant, nullptr);
            const ConvTapsKernel* k = v ? conv_taps_kernel(v->name) : nullptr;
            if (!k) return SHFLBW_ERR_UNSUPPORTED;
            ChwbTapArgs t;
            fill_spmm_launch_args(&state->spmm, v->BN, &t);
            t.B = a.in;
            t.store_mode = result_store_mode(t.D, t.M, t.ldd, bytes_of_b_and_c(t), stores_half_lines(state->brow, v->BN), false);
            t.alternate = 0;
            t.batch = a.B, t.in_h = a.H, t.in_w = a.W;
            t.taps_r = a.R, t.taps_s = a.S, t.stride = (int)chwb_stride(a.H, a.W, a.R, a.S, a.stride);
            t.magic_batch = udiv_magic(a.B), t.magic_w = udiv_magic(a.W);
            t.row_bits = 0;
            for (int r = 0; r < a.R; r++) t.row_bits |= 1u << (r * a.S);
            t.in_bytes = (unsigned)((size_t)a.C * a.H * a.W * a.B * 2);
            if (t.X > 0) e = k->launch(t, (hipStream_t)stream);
            if (e == hipSuccess) return SHFLBW_OK;
            set_error("spconv_exec: launch failed: %s", hipGetErrorString(e));
            return SHFLBW_ERR_HIP;
        }
        const ConvChwbKernel* k = conv_chwb_kernel(state->brow, state->middle_tile_cols, 0, 0, 0);
        if (!k) return SHFLBW_ERR_UNSUPPORTED;
        const bool nhwc = state->variant == FORM_BPLANES;
        e = nhwc ? launch_nhwc_to_planes(a, (half_t*)state->planes, state->plane_rows, state->plane_cols,
                                         state->plane_pitch, 1, (hipStream_t)stream, 1)
                 : launch_chwb_to_planes(a.in, (half_t*)state->planes, a.B, a.H, a.W, a.C, a.R, a.S, a.stride,
                                         state->plane_rows, state->plane_cols, state->plane_pitch, (hipStream_t)stream);
        SpmmLaunchArgs m;
        fill_spmm_launch_args(&state->spmm, k->BN, &m);
        m.alternate = 0;
        m.ldd = a.Ho * a.Wo * a.B;                  // a row of the result: one filter, Ho x Wo x B values
        m.store_mode = result_store_mode(m.D, m.M, m.ldd, bytes_of_b_and_c(m), stores_half_lines(state->brow, k->BN), nhwc);
        m.dmap_row = state->plane_cols * a.B;       // columns of the GEMM per row of the padded output grid
        m.dmap_valid = a.Wo * a.B;                  // ... of which the first Wo x B are output values
        m.dmap_magic = udiv_magic(m.dmap_row);
        if (e == hipSuccess && m.X > 0) e = k->launch(m, (hipStream_t)stream);
        if (e == hipSuccess && nhwc) // result_fm[f][(ho, wo, img)] -> OFMap[img][ho][wo][f]
            e = launch_planes_to_nhwc((const half_t*)state->result_fm, a.out, a.F, a.Ho * a.Wo * a.B, a.B, a.Ho, a.Wo,
                                      a.Ho, a.Wo, (hipStream_t)stream, 1);
    } else if (state->variant == FORM_FUSED) {
        const ConvXcdKernel* k = conv_xcd_kernel(state->brow);
        if (!k || state->xcds <= 0 || state->cols_per_xcd <= 0) return SHFLBW_ERR_UNSUPPORTED;
        SpmmLaunchArgs m;
        fill_spmm_launch_args(&state->spmm, k->BN, &m);
        if (m.X == 0) return SHFLBW_OK;
        m.alternate = 0; // a slab is far smaller than an L2
        m.ldd = state->cols_per_xcd;
        const int s = a.stride, nx = state->xcds, cx = state->cols_per_xcd;
        ConvXcdArgs c;
        c.g = PlaneGeom{a.B, a.H, a.W, a.C, s, a.pad_h, a.pad_w, state->plane_rows, state->plane_cols, state->plane_pitch, 1, 0, {}, 1};
        if (!fill_wanted_planes(c.g, a.R, a.S)) return SHFLBW_ERR_UNSUPPORTED;
        c.in = a.in;
        c.out = a.out;
        c.nx = nx, c.cx = cx, c.ncols = state->ncols;
        c.max_shift = (((a.R - 1) / s) * state->plane_cols + (a.S - 1) / s) * a.B;
        c.slabs = (half_t*)state->planes;
        c.slab_elems = up256((size_t)(s * s * a.C + 1) * state->plane_pitch * 2) / 2;
        c.fm = (half_t*)state->result_fm;
        c.fm_elems = up256((size_t)a.F * cx * 2) / 2;
        c.sync = (int*)state->sync;
        c.F = a.F, c.Ho = a.Ho, c.Wo = a.Wo;
        const int workers = std::max(1, m.num_cus / nx);
        const int n_x = std::min(cx, state->ncols); // the columns of a full XCD
        pick_chunk((a.C + 63) / 64, (n_x + c.max_shift + 63) / 64 * c.g.nwanted, workers, &c.ct, &c.pt, &c.ch_chunks);
        pick_chunk((a.F + 63) / 64, (n_x + 63) / 64, workers, &c.ft, &c.mt, &c.f_chunks);
        c.magic_b = udiv_magic(a.B);
        c.magic_pw = udiv_magic(state->plane_cols);
        c.spin_ticks = 20000000; // 0.2 s
        c.patience = state->patience_ticks > 0 ? state->patience_ticks : state->patience_ticks < 0 ? 1 : 5000;
        c.late_ticks = state->patience_ticks < 0 ? std::min(-state->patience_ticks, 10000) : 0;
        c.debug = 0;
#ifdef SHFLBW_CONV_STAMPS
        if (const char* dbg = getenv("SHFLBW_CONV_DEBUG")) c.debug = atoi(dbg);
#endif
        e = k->launch(m, c, (hipStream_t)stream);
    } else if (state->variant == FORM_PLANES) {
        e = launch_nhwc_to_planes(a, (half_t*)state->planes, state->plane_rows, state->plane_cols, state->plane_pitch,
                                  state->plane_copies, (hipStream_t)stream);
        if (e == hipSuccess) {
            int rc = shflbw_spmm_exec(&state->spmm, stream);
            if (rc != SHFLBW_OK) return rc;
            e = launch_planes_to_nhwc((const half_t*)state->result_fm, a.out, a.F, state->np, a.B, state->plane_rows,
                                      state->plane_cols, a.Ho, a.Wo, (hipStream_t)stream);
        }
    } else {
        const SpconvVariant* v = find_spconv_variant(state->brow, 0, nullptr); // the direct kernel of this block size
        if (!v) return SHFLBW_ERR_UNSUPPORTED;
        e = v->launch(a, (hipStream_t)stream);
    }
    if (e != hipSuccess) {
        set_error("spconv_exec: launch failed: %s", hipGetErrorString(e));
        return SHFLBW_ERR_HIP;
    }
    return SHFLBW_OK;
}

int shflbw_spconv_check(const shflbw_spconv_state* state)
{
    if (!state || !state->init_success) {
        set_error("spconv_check: state was not initialised successfully");
        return SHFLBW_ERR_STATE;
    }
    if (state->variant != FORM_FUSED) return SHFLBW_OK;
    int flag = 0;
    SHFLBW_HIP_TRY(hipMemcpy(&flag, state->sync, sizeof(int), hipMemcpyDeviceToHost)); // waits for the device
    if (flag != 0) {
        // leave the scratch as a fresh one: no counter may keep what the failed launch left in it
        SHFLBW_HIP_TRY(hipMemset(state->sync, 0, (size_t)conv_xcd_sync_lines(state->xcds) * SYNC_LINE * sizeof(int)));
        set_error(flag == 1 ? "spconv_check: the workgroups of a fused launch were not dealt to the XCDs the way init had checked; results are invalid"
                            : "spconv_check: a wait between the phases of the fused form ran out of time; results are invalid");
        return SHFLBW_ERR_HIP;
    }
    return SHFLBW_OK;
}

// ---------------------------------------------------------------------------------------------------
// The entry point that allocates nothing: the scratch of the plane form in a fixed device array.
// `scratch` below is only the host-side handle of the symbol; the device address of each GPU's copy
// comes from hipGetSymbolAddress, once per device, and only that address is handed to kernels.
// ---------------------------------------------------------------------------------------------------
} // extern "C"

static __device__ __align__(256) unsigned char scratch[SHFLBW_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_static_lock;
void* g_static_addr[kMaxDevices] = {};

// device address of this GPU's copy of `scratch` (looked up on the first call with that device current)
int static_scratch_address(char** out)
{
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        set_error("spconv_exec_static: cannot tell the current device");
        return SHFLBW_ERR_HIP;
    }
    std::lock_guard<std::mutex> guard(g_static_lock);
    if (!g_static_addr[dev]) {
        void* ptr = nullptr;
        hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            set_error("spconv_exec_static: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
            return SHFLBW_ERR_HIP;
        }
        g_static_addr[dev] = ptr;
    }
    *out = (char*)g_static_addr[dev];
    return SHFLBW_OK;
}
} // namespace

extern "C" {

int shflbw_spconv_exec_static(const shflbw_weight* f, int B, int H, int W, int stride, const void* IFMap, void* OFMap,
                              void* stream)
{
    shflbw_spconv_state st;
    int rc = spconv_fill_state(&st, f, B, H, W, stride, IFMap, OFMap, FORM_PLANES);
    if (rc != SHFLBW_OK) return rc;
    PlaneForm g;
    if ((rc = plane_form_geometry(f, B, H, W, stride, &g)) != SHFLBW_OK) return rc;
    if (g.total_bytes() > (size_t)SHFLBW_STATIC_SCRATCH_BYTES) {
        set_error("spconv_exec_static: this problem needs %zu bytes of scratch, the fixed array holds %zu", g.total_bytes(),
                  (size_t)SHFLBW_STATIC_SCRATCH_BYTES);
        return SHFLBW_ERR_CAPACITY;
    }
    char* base = nullptr;
    if ((rc = static_scratch_address(&base)) != SHFLBW_OK) return rc;
    // Nothing in the array has to start at zero: the layout pass writes every plane position a pixel's taps
    // read (zeros outside the image), the rest only feeds plane positions that are no output pixel.
    int* ids = (int*)(base + g.planes_bytes + g.dm_bytes);
    int* ids_pm = (int*)(base + g.planes_bytes + g.dm_bytes + g.ids_bytes);
    if ((rc = bind_plane_form(&st, f, g, base, base + g.planes_bytes, ids, ids_pm)) != SHFLBW_OK) return rc;
    hipError_t e = launch_plane_ids((const int*)f->d_packed_indices, ids, ids_pm, (int)g.slots, f->C, f->S, stride, g.PW,
                                    (int)g.pitch, g.copies, (int)(g.rows * g.pitch), (half_t*)base, (hipStream_t)stream);
    if (e != hipSuccess) {
        set_error("spconv_exec_static: id launch failed: %s", hipGetErrorString(e));
        return SHFLBW_ERR_HIP;
    }
    return shflbw_spconv_exec(&st, stream);
}

static const char* const g_spconv_forms[FORM_COUNT] = {
    "planes+spmm+transpose",  // 0: NHWC -> channel-major planes, SpMM gather with tap offsets, transpose to NHWC: three launches
    "direct",                 // 1: one kernel, im2col gather from NHWC in the tile loads
    "bplanes+spmm+transpose", // 2: NHWC tensors, planes and result with the batch innermost (batch a multiple of 8): three launches
    "bplanes-fused",          // 3: the steps of form 2 in one persistent launch, every XCD on its own columns
    "chwb",                   // 4: the reference's batch-innermost tensors (shflbw_spconv_init_chwb only): one launch over the input; padded copy and SpMM where its ids do not fit
    "patch",                  // 5: one launch, the input patch of a workgroup's pixels in LDS, channel-major
};

int shflbw_spconv_variant_count(void) { return FORM_COUNT; }

const char* shflbw_spconv_variant_name(int variant)
{
    return variant >= 0 && variant < FORM_COUNT ? g_spconv_forms[variant] : "";
}

int shflbw_weight_release_scratch(shflbw_weight* w)
{
    if (!w) return SHFLBW_ERR_INVALID;
    std::lock_guard<std::mutex> guard(w->scratch_lock);
    release_conv_scratch(w);
    return SHFLBW_OK;
}

int shflbw_weight_scratch_bytes(const shflbw_weight* w, size_t* bytes, int* buffers)
{
    if (!w) return SHFLBW_ERR_INVALID;
    shflbw_weight* fw = const_cast<shflbw_weight*>(w);
    std::lock_guard<std::mutex> guard(fw->scratch_lock);
    size_t total = 0;
    for (auto& e : w->conv_ids) total += e.bytes;
    for (auto& e : w->conv_bulk) total += e.bytes;
    for (auto& e : w->patch_images) total += e.bytes;
    int places = 0; // those that are no part of an image
    for (auto& e : w->patch_places) total += e.bytes, places += e.ptr != nullptr;
    if (bytes) *bytes = total;
    if (buffers) *buffers = (int)(w->conv_ids.size() + w->conv_bulk.size() + w->patch_images.size()) + places;
    return SHFLBW_OK;
}

void shflbw_abi_sizes(size_t* spmm_state_bytes, size_t* spconv_state_bytes)
{
    if (spmm_state_bytes) *spmm_state_bytes = sizeof(shflbw_spmm_state);
    if (spconv_state_bytes) *spconv_state_bytes = sizeof(shflbw_spconv_state);
}

int shflbw_device_info(int* compute_units, int* clock_khz, size_t* lds_bytes, char* arch, size_t arch_cap)
{
    int dev = 0;
    SHFLBW_HIP_TRY(hipGetDevice(&dev));
    hipDeviceProp_t p;
    SHFLBW_HIP_TRY(hipGetDeviceProperties(&p, dev));
    if (compute_units) *compute_units = p.multiProcessorCount;
    if (clock_khz) *clock_khz = p.clockRate;
    if (lds_bytes) *lds_bytes = p.sharedMemPerBlock;
    if (arch && arch_cap) {
        strncpy(arch, p.gcnArchName, arch_cap - 1);
        arch[arch_cap - 1] = 0;
    }
    return SHFLBW_OK;
}

} // extern "C"
