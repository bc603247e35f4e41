// Launch-side description of the native SpMM tile variants (host + device shared).
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <initializer_list>

#include "kernel_common.h"
#include "shflbw.h"

namespace shflbw {

// The C term of a launch: none (beta == 0), or how C is read
enum CTerm { C_NONE = 0, C_CACHED = 1, C_STREAMED = 2 };

struct SpmmLaunchArgs {
    int M, N, K;
    int X;       // row panels = M / V
    unsigned magic_x; // udiv_magic of X
    unsigned magic_halves[2]; // udiv_magic of the panels of either part (launcher, where they are taken apart)
    int n_tiles; // column tiles, filled by the launcher
    unsigned magic_tiles; // split kernel: udiv_magic of n_tiles; slab kernel: of what job numbers are cut by, n_tiles or slab_chunks (launcher)
    int split_shift;      // split kernel only: log2 of the 32-row blocks of a panel (launcher)
    const half8_t* packedA; // private image: A fragments in register order
    const int* kidx;        // private image: kept column ids, 64-slot padded per panel
    const int* kidx_pm;     // same ids, each 64-slot group reordered producer-major: [16p + 4j + r] = [16j + 4p + r]
    const int* slab_ids;    // slab kernel only: the ids as LDS offsets of slab rows, [group][pair of slots][step][2]
    int groups;             // 64-slot groups of all panels
    int slab_chunks;        // slab kernel only: the panels are dealt to this many workgroups per column tile (launcher)
    int slab_panels;        // ... the panels of a chunk (launcher)
    int slab_by_chunk;      // slab kernel only: jobs of one chunk of panels lie side by side instead of those of one column tile (launcher)
    const int* panel_desc;  // private image: per panel {MFMA k16 steps = ceil(nnz/16), first 64-slot group}
    const int* row_ids;     // M, or null when rows are not permuted
    const half_t* B;
    const void* zero_row;   // 1 KiB of zeros on the device: what the padding slots (id -1) of a panel's last group gather where B has no descriptor
    int ldb_bytes;          // bytes between rows of B one id apart (N * 2 for a dense row-major B)
    const half_t* C;
    half_t* D;
    int ldd;                // values between two rows of C and D (N for the SpMM)
    int store_mode;         // a StoreMode: how D is stored, see result_store_mode (slab kernel: slab_plan)
    int dmap_row, dmap_valid; // batch-innermost convolution only: see output_column()
    unsigned dmap_magic;      // udiv magic of dmap_row
    float alpha, beta;
    int num_cus; // compute units of the device (persistent kernels size their grid with it)
    int alternate; // role-split kernels: walk every second tile of a workgroup from its last stage to its first
                   // (pays when the rows of B under one column tile do not fit the XCD's L2; in halves too, where a workgroup's next
                   // tile is another column tile of the same panels, whose A it then finds: us, one way / alternating: 8192 x
                   // 8192 x 16384, 0.07 226 / 222, with C 271 / 259, 5120 x 8192 x 16384, 0.11 198 / 189, with C 217 / 208)
    int half_panels; // panels of the first of two parts of about the same work, 0: no such cut (spmm_half_panels).  Stands last: eight
                     // bytes more in front of the pointers cost the smallest products 0.18 us (1024^3, density 0.25: 4.24 / 4.42),
                     // the loads of the arguments fall into other lines
};

// Convolution over batch-innermost tensors that gathers from the input itself (B points to it): the columns of the GEMM
// are the output positions (ho, wo, b), a kept column is a channel plane and a tap, ids as chwb_tap_id() packs them.
struct ChwbTapArgs : SpmmLaunchArgs {
    int batch, in_h, in_w;      // batch, a multiple of 8; H and W bound input and output alike
    int taps_r, taps_s, stride; // R * S <= CHWB_MAX_TAPS
    unsigned magic_batch, magic_w; // udiv_magic of batch and in_w
    unsigned row_bits;          // bits r * S for all r < R
    unsigned in_bytes;          // of the whole input, below 2^31
};
constexpr int CHWB_MAX_TAPS = 31;  // a lane keeps one bit per tap; bit 31 is that of the padding slots, which no lane reads
// units of 16 bytes from the lane's own position at tap (0, 0) of channel 0, and the tap
constexpr int chwb_tap_id(unsigned units16, unsigned tap) { return (int)(units16 * 32u + tap); }

// Raises the dynamic-LDS limit of kernels, once per device (`raised`: one bit each): an initialisation makes no call into the
// driver for a limit that is already raised.
inline hipError_t raise_lds_limit(std::atomic<unsigned long long>& raised, std::initializer_list<const void*> kernels, int bytes)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const unsigned long long bit = dev < 64 ? 1ull << dev : 0;
    if (raised.load(std::memory_order_acquire) & bit) return hipSuccess;
    for (const void* f : kernels)
        if ((e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes)) != hipSuccess) return e;
    raised.fetch_or(bit, std::memory_order_release);
    return hipSuccess;
}

struct SpmmVariant {
    int V;           // block size (rows per panel)
    int BN;          // output columns per workgroup
    int threads;     // workgroup size
    int lds_bytes;   // dynamic LDS
    const char* name;
    hipError_t (*launch)(const SpmmLaunchArgs&, hipStream_t);
    hipError_t (*prepare)(const SpmmLaunchArgs&); // raises the dynamic-LDS limit of the kernels that `launch` may take (M, N, X are set)
    int max_k;               // 0, or the most columns of A the variant takes (it holds all rows of B in LDS)
    int per_cu;              // role-split variants: workgroups a compute unit holds at once
};

const SpmmVariant* spmm_variants(int* count);

// How the slab kernel deals X panels (groups of 64 slots in all) under n_tiles column tiles to workgroups: at least as many chunks
// as keep the panels of one wave within the rows it has registers for; then the number that takes the least rounds * (slab + panels
// of a wave), of the most that one, two and three rounds of the compute units have room for (us, from the phases of a wave).
// 33728 x 1100 x 2112, block height 32: 33 tiles x 9 chunks were two rounds, the second nearly empty, 91 us; 15 chunks 66.
constexpr int SLAB_WAVES = 8;          // of a workgroup
constexpr int SLAB_WAVE_ROWS = 8 * 64; // rows of D a wave holds the places of
struct SlabDeal {
    int chunks, rounds, wave_panels;
};
inline SlabDeal slab_deal(int V, int X, int K, int groups, int n_tiles, int cus)
{
    const int least = (X * V + SLAB_WAVES * SLAB_WAVE_ROWS - 1) / (SLAB_WAVES * SLAB_WAVE_ROWS);
    const double batches = 2.0 * groups / X; // of 32 slots, per panel
    const double t_slab = 1.0 + 1.5e-3 * K, t_panel = V == 16 ? 0.30 + 0.12 * batches : 0.45 + 0.21 * batches;
    SlabDeal best{};
    double best_t = 0;
    for (int r = 1; r <= 3; r++) {
        const int most = cus * r / n_tiles, at_least = most > least ? most : least;
        SlabDeal d;
        d.chunks = at_least < 1 ? 1 : at_least > X ? X : at_least;
        d.rounds = (int)(((long)n_tiles * d.chunks + 7) / 8 * 8 + cus - 1) / cus;
        d.wave_panels = ((X + d.chunks - 1) / d.chunks + SLAB_WAVES - 1) / SLAB_WAVES;
        const double t = d.rounds * (t_slab + d.wave_panels * t_panel);
        if (r == 1 || t < best_t * 0.95) best_t = t, best = d;
    }
    return best;
}

// Bytes of B, C and D from which on three problems in turn leave the Infinity Cache (256 MB).
constexpr size_t STORE_MERGE_BYTES = 80u << 20;
inline size_t bytes_of_b_and_c(const SpmmLaunchArgs& a) { return (size_t)a.K * a.ldb_bytes + (a.beta != 0.f ? (size_t)a.M * a.ldd * 2 : 0); }

// How the slab kernel stores D, as result_store_mode for the role-split kernels.  us, through / merged / streamed, the better order of
// jobs each: whole lines, block height 32, density 0.2: 4096 x 1024 x 4096 17.0 / 18.1 / 17.2, 8192 x 768 x 8192 62 / 62 / 48; block height 16,
// 33728 x 777 x 1024 22.1 / 24.3 / 22.4, 20000 x 1000 x 6016 85 / 89 / 69.  Parts of lines: 8192 x 777 x 3000 (49 MB) 19.4 / 21.0 / 32, block
// height 32, 33728 x 1100 x 2104 136 / 123 / 121, 16: 20000 x 1000 x 6000 145 / 101 / 125; merged / through over 191 drawn problems: 0.88 by
// this rule, 1.02 at worst, with the line at D >= 64 MB, as before, 0.89 and 1.15 (16592 x 76 x 2848, block height 16, 95 MB: 21.7 and 24.1 us).
inline StoreMode slab_store_mode(const void* D, int rows, int ldd, size_t others)
{
    const size_t bytes = (size_t)rows * (size_t)ldd * 2;
    if ((((uintptr_t)D | ((uintptr_t)ldd * 2)) & 127) != 0) return bytes + others >= STORE_MERGE_BYTES ? STORE_MERGE : STORE_THROUGH;
    return bytes >= 96u << 20 ? STORE_STREAM : STORE_THROUGH;
}

// Whether the panels are cut in two halves that the XCDs work on apart; S: workgroups of an XCD.  With all panels under one column tile
// after the other every XCD reads the whole of A once per column tile, from the Infinity Cache where A exceeds the L2, and its
// workgroups store pieces of one column tile at a time.  In halves it reads half of A and is on two column tiles at a time, or its
// neighbours are on other ones, for a second trip of B.  That helps large results of block height 128 with an A of at most 10 MB, half of
// which stays in an L2 for the most part.  Times of halves over whole panels, 436 problems, from 24 panels on where nothing else is said:
//  * where A is longer than 6 MB and there are at most 40 panels, two column tiles to a round: 0.95 to 1.04, 0.988 on average (4096 x
//    2775 x 14592, density 0.32 120 us / 113, 3456 x 2890 x 20544, 0.26 184 / 175, 4608 x 4960 x 27840, 0.15, with C 272 / 283).  41 to 47
//    panels 0.94 to 1.04, 1.00; from 48 on 0.95 to 1.13, 1.03; an A of 4.5 to 6 MB 0.89 to 1.04, 0.99, above 10 MB 0.97 to 1.03, 0.99; 14
//    to 23 panels, three column tiles and more, 0.96 to 1.05, 0.995; below that the larger part decides;
//  * where the pitch of D is a multiple of 32 KiB, which puts a column tile's pieces of all rows into the same few channels of the
//    memory; in halves the workgroups of an XCD, or those of its neighbours, are on other column tiles.  An A longer than 6 MB without C
//    0.91 to 1.02, 0.97, with C 0.88 to 1.01, 0.955 (8192 x 4500 x 16384, 0.085, with C 234 us / 214, without 178 / 173; 16384 x 4096 x 16384,
//    0.059 367 / 339 and 268 / 252; above 10 MB 0.93 to 1.06, 0.98); a shorter one with C and permuted rows 0.76 to 1.06, 0.89 (14336 x
//    2048 x 16384, 0.027 274 / 218), rows not permuted 0.91 to 1.13, 0.985, without C 0.71 to 1.11, 0.94; below 24 panels 0.85 to 1.11, 0.98.
inline bool panel_halves(const SpmmLaunchArgs& a, int S)
{
    const size_t a_bytes = (size_t)a.groups * 64 * (a.M / a.X) * 2;
    if (a.store_mode != STORE_STREAM || a.half_panels <= 0 || a.half_panels >= a.X || 4 * a.X < 3 * S || a_bytes > 10u << 20) return false;
    const bool long_a = a_bytes > 6u << 20;
    if ((size_t)a.ldd * 2 % (32u << 10) == 0) return long_a || (a.beta != 0.f && a.row_ids != nullptr);
    return long_a && 4 * a.X <= 5 * S;
}

// Whether C is streamed past the caches: where D is, and B, C and D are twice the Infinity Cache, nothing of C lasts until a next pass. us,
// cached / streamed: block height 64, 8192 x 4096 x 16384, density 0.1 (670 MB) 256 / 233, 16384 x 4096 x 8192, 0.05 (604 MB) 177 / 170,
// 14144 x 1186 x 13824, 0.16 (815 MB) 239 / 230; 128: 32768 x 2048 x 4096, 0.1 (553 MB) 146 / 143; but 64, 9152 x 1339 x 12288, 0.17 (482
// MB) 142 / 146, 11584 x 1908 x 9216, 0.13 (462 MB) 134 / 146, and D in parts of lines, 128, 17280 x 6409 x 13928, 0.025 342 / 369.  50
// drawn problems above the line, over three sets of operands in turn 0.90 to 1.00 times as long streamed, over one set 0.90 to 1.03 (9920 x
// 120 x 14272 119 / 123); below it, from 400 MB, 0.95 to 1.01 and 0.94 to 1.34.
inline bool streams_c(const SpmmLaunchArgs& a)
{
    return a.store_mode == STORE_STREAM && bytes_of_b_and_c(a) + (size_t)a.M * a.ldd * 2 >= 512u << 20;
}

// Launch arguments of the SpMM kernels from a state; BN is the tile width of the kernel that will run.
void fill_spmm_launch_args(const shflbw_spmm_state* state, int BN, SpmmLaunchArgs* out);

// device address of the library's row of zeros on the current device (looked up once per device); null on failure
const void* spmm_zero_row();

} // namespace shflbw
