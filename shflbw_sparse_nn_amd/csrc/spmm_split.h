// Split form of the SpMM for few columns (decoding: N counts the tokens of one step).  The role-split kernel gives a panel to
// one workgroup whose four consumers split the columns: at N = 8 three of them and most of every gather work for padding,
// and M / V workgroups - 16 of them for a 2048-row weight of block height 128 - leave the chip idle while each walks all
// kept vectors of its panel.  What bounds such a call is the weight, read once, and latency.  So here the waves split the
// kept vectors: a workgroup owns 32 output rows (16 for block height 16; a panel of 64 or 128 rows is two or four
// workgroups) and 32 or 64 columns, each of its 8 or 16 waves runs a contiguous share of the kept vectors through MFMAs
// from an LDS ring of its own - no barrier before the partial sums (fp32, added in a fixed order) meet in LDS.
// Replaces, for such shapes, the reference's main loop (block_sparse/spmm/blockwise_kernel.h:108-294).
#pragma once
#include <type_traits>

#include "kernel_common.h"
#include "spmm_launch.h"

namespace shflbw {

// NBK: 32-column blocks of a workgroup's columns; V16: block height 16 (16x16x32 tiles, 32 slots per step)
template <bool V16, int NBK>
struct SpmmSplitCfg {
    static constexpr int RB = V16 ? 16 : 32;              // output rows of a workgroup
    static constexpr int SLOTS = V16 ? 32 : 16;           // kept vectors per step
    static constexpr int BN = 32 * NBK;
    static constexpr int ROWB = BN * 2;                   // bytes of a gathered row
    static constexpr int B_BYTES = SLOTS * ROWB;
    static constexpr int STEP_BYTES = B_BYTES + 1024;     // gathered rows and one A fragment
    static constexpr int J = B_BYTES / 1024;              // gather instructions per step
    static constexpr int PPR = ROWB / 16;                 // 16-byte pieces per row
    static constexpr int RPI = 64 / PPR;                  // rows per gather instruction
    static constexpr int OPS = J + 2;                     // copies per step: rows, A fragment, ids
    static constexpr int NST = STEP_BYTES <= 2048 ? 4 : 3; // steps in flight: as many as fit the LDS
    static constexpr int ID_BYTES = 256;                  // ids of a step in LDS (one copy brings 64, the first SLOTS are used)
    static constexpr int WAVE_BYTES = NST * (STEP_BYTES + ID_BYTES);
    static constexpr int RED_ROWB = (BN + 4) * 4;         // row of partial sums, padded
    static constexpr int RED_WAVE_BYTES = RB * RED_ROWB;
    static constexpr int OUT_THREADS = RB * BN / 4;       // four columns each
    static constexpr int MAX_WAVES = 16;
    static constexpr int lds_bytes(int waves) { return waves * (WAVE_BYTES > RED_WAVE_BYTES ? WAVE_BYTES : RED_WAVE_BYTES); }
    static_assert(lds_bytes(MAX_WAVES) <= 160 * 1024, "LDS budget of a gfx950 compute unit");
    static_assert(!V16 || NBK == 1, "see split_wide_tiles()");
    static_assert(OUT_THREADS <= 8 * 64, "the smallest workgroup stores its result in one pass");
    static_assert((NST - 1) * OPS < 64, "vmcnt is a 6-bit counter");

    // 32-byte unit of a gathered row where logical unit u lies: the rows one transposing read touches spread over the banks
    __device__ __forceinline__ static constexpr int unit_pos(int u, int row)
    {
        return NBK == 2 ? u ^ (((row >> 1) & 1) << 1) : V16 ? u ^ ((row >> 3) & 1) : u;
    }
};

template <bool V16, int NBK>
__global__ void __launch_bounds__((SpmmSplitCfg<V16, NBK>::MAX_WAVES * 64)) spmm_shflbw_split_kernel(SpmmLaunchArgs a)
{
    using Cfg = SpmmSplitCfg<V16, NBK>;
    constexpr int RB = Cfg::RB, SLOTS = Cfg::SLOTS, ROWB = Cfg::ROWB, J = Cfg::J, NST = Cfg::NST, OPS = Cfg::OPS, PPR = Cfg::PPR;
    extern __shared__ __attribute__((aligned(1024))) char lds_raw[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(SHFLBW_LDS char*)lds_raw;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nw = blockDim.x >> 6;
    const int N = a.N, V = a.M / a.X;
    // the column tiles of a row block lie on one XCD (workgroup ids go round the XCDs), which reads its fragments once
    const int q = blockIdx.x >> 3;
    const int blk = q / a.n_tiles * 8 + (blockIdx.x & 7);
    const int n0 = q % a.n_tiles * Cfg::BN;
    if (blk * RB >= a.M) return;
    const int panel = blk * RB / V;
    const int mb = V16 ? 0 : blk - panel * (V / 32), mbs = V16 ? 1 : V / 32;
    const int2_t pd = ((const SHFLBW_CONST int2_t*)(uintptr_t)a.panel_desc)[panel]; // {k16 steps, first 64-slot group}
    const int steps = V16 ? (pd.x + 1) >> 1 : pd.x;
    const int per = (steps + nw - 1) / nw; // steps of a wave
    const int s0 = min(steps, wave * per), cnt = min(steps, s0 + per) - s0;

    // what this thread stores: four columns of one row
    const int orr = tid / (Cfg::BN / 4), oc = n0 + tid % (Cfg::BN / 4) * 4;
    const bool out = tid < Cfg::OUT_THREADS && oc < N;
    int orow = blk * RB + orr;
    if (out && a.row_ids) orow = a.row_ids[orow];

    // ---- this wave's ring: steps of gathered rows and a fragment, then the ids
    const uint32_t ring = lds0 + wave * Cfg::WAVE_BYTES, idring = ring + NST * Cfg::STEP_BYTES;
    int grow[J], gcol[J]; // row of the step and column (bytes) that this lane fetches with gather instruction j
#pragma unroll
    for (int j = 0; j < J; j++) {
        grow[j] = j * Cfg::RPI + lane / PPR;
        const int pos = lane % PPR;
        const int col = n0 + Cfg::unit_pos(pos >> 1, grow[j]) * 16 + (pos & 1) * 8;
        gcol[j] = (col < N ? col : n0) * 2; // columns past N are never stored
    }
    const int slots = ((pd.x + 3) >> 2) * 64; // of the panel, padded
    const int* ids = a.kidx + (size_t)pd.y * 64;
    const char* frags = (const char*)a.packedA + (size_t)pd.y * (64 * V * 2) + mb * 1024 + lane * 16;
    auto copy_ids = [&](int t, int slot) __attribute__((always_inline)) { // past the last step: ids nobody uses
        global_to_lds_4B(ids + min((s0 + t) * SLOTS + lane, slots - 1), idring + slot * Cfg::ID_BYTES);
    };
    auto issue = [&](int t, int slot) __attribute__((always_inline)) {
        const uint32_t st = ring + slot * Cfg::STEP_BYTES;
        int id[J];
#pragma unroll
        for (int j = 0; j < J; j++) id[j] = *(SHFLBW_LDS int*)(uintptr_t)(idring + slot * Cfg::ID_BYTES + grow[j] * 4);
        // the ids are in registers before the copy below overwrites them
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int j = 0; j < J; j++) asm volatile("" : "+v"(id[j]) : : "memory");
#pragma unroll
        for (int j = 0; j < J; j++) {
            // a padding slot (id -1) gathers 16 bytes per lane of the row of zeros
            const char* src = id[j] < 0 ? (const char*)a.zero_row + lane * 16
                                        : (const char*)a.B + (size_t)id[j] * (uint32_t)a.ldb_bytes + gcol[j];
            global_to_lds_16B(src, st + j * 1024);
        }
        global_to_lds_16B(frags + (size_t)(s0 + t) * mbs * 1024, st + Cfg::B_BYTES);
        copy_ids(t + NST, slot);
    };

    // ---- transposing reads: a group of 16 lanes reads 4 rows x 32 bytes
    constexpr int NB = V16 ? 2 * NBK : NBK; // accumulator blocks
    const int li = lane & 15;
    const int r0 = 8 * (V16 ? lane >> 4 : lane >> 5) + (li >> 2);
    uint32_t blo[NB], bhi[NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        const int u = V16 ? nb : nb * 2 + ((lane >> 4) & 1);
        blo[nb] = (uint32_t)(r0 * ROWB + (Cfg::unit_pos(u, r0) << 5) + ((li & 3) << 3));
        bhi[nb] = (uint32_t)((r0 + 4) * ROWB + (Cfg::unit_pos(u, r0 + 4) << 5) + ((li & 3) << 3));
    }
    using acc_t = typename std::conditional<V16, float4_t, float16_t>::type;
    acc_t acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; nb++)
#pragma unroll
        for (int i = 0; i < (V16 ? 4 : 16); i++) acc[nb][i] = 0.f;

    if (cnt > 0) {
#pragma unroll
        for (int t = 0; t < NST; t++) copy_ids(t, t);
        wait_vmcnt_fence<0>();
#pragma unroll
        for (int t = 0; t < NST; t++)
            if (t < cnt) issue(t, t);
        int slot = 0;
        for (int t = 0; t < cnt; t++) {
            // step t and the ids issued with it have arrived; up to NST - 1 younger steps stay in flight
            if (t + NST <= cnt)
                wait_vmcnt_fence<(NST - 1) * OPS>();
            else
                wait_vmcnt_fence<0>();
            const uint32_t st = ring + slot * Cfg::STEP_BYTES;
            half8_t af = *(SHFLBW_LDS half8_t*)(uintptr_t)(st + Cfg::B_BYTES + lane * 16);
            half8_t bf[NB];
#pragma unroll
            for (int nb = 0; nb < NB; nb++) {
                const half4_t lo = lds_read_tr16(st + blo[nb]);
                const half4_t hi = lds_read_tr16(st + bhi[nb]);
                bf[nb] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            }
            // everything read before the slot is filled again
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            asm volatile("" : "+v"(af) : : "memory");
#pragma unroll
            for (int nb = 0; nb < NB; nb++) asm volatile("" : "+v"(bf[nb]) : : "memory");
            if (t + NST < cnt) issue(t + NST, slot);
#pragma unroll
            for (int nb = 0; nb < NB; nb++) {
                if constexpr (V16)
                    acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[nb], af, acc[nb], 0, 0, 0);
                else
                    acc[nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bf[nb], af, acc[nb], 0, 0, 0);
            }
            slot = slot + 1 == NST ? 0 : slot + 1;
        }
    }
    const float alpha = a.alpha, beta = a.beta;
    half4_t c = {0, 0, 0, 0};
    if (beta != 0.f && out) c = *(const half4_t*)(a.C + (size_t)orow * a.ldd + oc);

    // ---- partial sums meet in LDS, over the rings: all copies into them have landed (also ids nobody uses)
    wait_vmcnt_fence<0>();
    __syncthreads();
    if (cnt > 0) {
        const uint32_t red = lds0 + wave * Cfg::RED_WAVE_BYTES + (lane & (RB - 1)) * Cfg::RED_ROWB;
#pragma unroll
        for (int nb = 0; nb < NB; nb++) {
            if constexpr (V16) {
                *(SHFLBW_LDS float4_t*)(uintptr_t)(red + (nb * 16 + (lane >> 4) * 4) * 4) = acc[nb];
            } else {
#pragma unroll
                for (int ig = 0; ig < 4; ig++)
                    *(SHFLBW_LDS float4_t*)(uintptr_t)(red + (nb * 32 + ig * 8 + (lane >> 5) * 4) * 4) =
                        float4_t{acc[nb][ig * 4], acc[nb][ig * 4 + 1], acc[nb][ig * 4 + 2], acc[nb][ig * 4 + 3]};
            }
        }
    }
    __syncthreads();
    if (!out) return;
    const int sums = per > 0 ? (steps + per - 1) / per : 0; // waves that had a step
    const uint32_t rd = lds0 + orr * Cfg::RED_ROWB + (oc - n0) * 4;
    float4_t s = {0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < sums; w++) s += *(SHFLBW_LDS float4_t*)(uintptr_t)(rd + w * Cfg::RED_WAVE_BYTES);
    half4_t h;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        h[e] = (half_t)scaled(s[e], alpha, beta != 0.f);
        if (beta != 0.f) h[e] = (half_t)((float)h[e] + beta * (float)c[e]);
    }
    *(half4_t*)(a.D + (size_t)orow * a.ldd + oc) = h;
}

template <bool V16, int NBK>
static hipError_t launch_split_n(const SpmmLaunchArgs& a, hipStream_t stream)
{
    using Cfg = SpmmSplitCfg<V16, NBK>;
    SpmmLaunchArgs b = a;
    b.n_tiles = (a.N + Cfg::BN - 1) / Cfg::BN;
    const long blocks = (a.M / Cfg::RB + 7) / 8 * 8, grid = blocks * b.n_tiles;
    if (grid > 0x7fffffffL) return hipErrorInvalidValue;
    // one workgroup per compute unit: as many waves as its LDS feeds; else two workgroups at a time
    const int waves = grid <= (a.num_cus > 0 ? a.num_cus : 256) ? Cfg::MAX_WAVES : 8;
    hipLaunchKernelGGL((spmm_shflbw_split_kernel<V16, NBK>), dim3((unsigned)grid), dim3(waves * 64), Cfg::lds_bytes(waves), stream, b);
    return hipGetLastError();
}

// 64-column tiles where 32-column ones would outnumber the compute units (two of those take as long per step and 0.3 us
// more per 64 columns).  Block height 16 has only the narrow ones: its wide step is 5 KiB, of which the LDS holds two
// dozen, and takes 2.2 times a narrow one.
static bool split_wide_tiles(const SpmmLaunchArgs& a)
{
    return a.X > 0 && a.M / a.X != 16 && a.N > 32 && (long)(a.M / 32) * ((a.N + 31) / 32) > (a.num_cus > 0 ? a.num_cus : 256);
}

template <bool V16>
static hipError_t launch_split(const SpmmLaunchArgs& a, hipStream_t stream)
{
    if (a.X <= 0 || a.M % a.X != 0 || a.N <= 0 || a.N % 8 != 0) return hipErrorInvalidValue;
    if constexpr (!V16)
        if (split_wide_tiles(a)) return launch_split_n<V16, 2>(a, stream);
    return launch_split_n<V16, 1>(a, stream);
}

template <bool V16, int NBK>
static hipError_t prepare_split_n()
{
    using Cfg = SpmmSplitCfg<V16, NBK>;
    static std::atomic<unsigned long long> raised{0};
    return raise_lds_limit(raised, {(const void*)spmm_shflbw_split_kernel<V16, NBK>}, Cfg::lds_bytes(Cfg::MAX_WAVES));
}

template <bool V16>
static hipError_t prepare_split(const SpmmLaunchArgs& a)
{
    if constexpr (!V16)
        if (split_wide_tiles(a)) return prepare_split_n<V16, 2>();
    return prepare_split_n<V16, 1>();
}

} // namespace shflbw
