// Patch form of the Shfl-BW convolution: NHWC in, NHWC out, one launch.
//
// The plane forms rewrite the input channel-major in memory and the result pixel-major: two passes over memory and
// two more launches around an SpMM that itself takes half of the time.  Here a workgroup owns 64 (or 32) output
// pixels and a set of filters:
//   1. it copies the input patch under its pixels (halo included) into LDS and transposes it on the way: one row
//      per channel, the four units of a position side by side in 8 bytes;
//   2. every wave streams the A fragments of its own row panels and the LDS offsets of their kept columns straight
//      into registers (several batches in flight) and reads its B fragments from the rows the offsets name
//      (transposing LDS reads; tap, stride and position are one added offset), MFMA, fp32 accumulators;
//   3. the fp16 results go through LDS (pixel rows, filters in output order) to whole runs of the NHWC output.
// What bounds it: the chain of these phases, with one workgroup per compute unit on layers of many channels.  16 x 14 x 14 x 512 ->
// 2048, 3 x 3, block height 64, density 0.1 (17.6 us; us after a wave's start): arguments 0.7, patch asked for until 1.9 (160 KB at the
// 64 bytes a clock of a compute unit) and in LDS at 3.5, products 4.4 near the matrix cores' rate (the A stream is level with them), the
// slowest wave 0.8 later, results to LDS 0.8, 2-byte stores of the permuted filters 3.5, bound by the pieces of 64 bytes that the L2s
// write (consecutive 2-byte stores: 2.0).  32 x 28 x 28 x 256 -> 512, stride 2, block height 32, density 0.3 (14.0 us): 0.7, 3.7, 4.8 (matrix
// cores 56 %, A stream 54 %, the rest LDS reads), 0.5, 0.4, 1.9.  On small layers launch, patch, first fragments and stores, a round trip
// each.
#include "spconv_patch.h"

#include <algorithm>
#include <type_traits>
#include <cmath>

namespace shflbw {

// RW: rows of a row unit - one row panel, half of one for block height 128
template <int RW>
struct ConvPatchCfg {
    static constexpr bool R16 = RW == 16;
    static constexpr int MBW = RW == 64 ? 2 : 1;     // A fragments per MFMA step
    static constexpr int STEPS = R16 ? 1 : 2;        // MFMA steps per batch of 32 slots
    static constexpr int NA = STEPS * MBW;           // A fragments per batch
    static constexpr int OPS = NA + 1;               // loads per batch
};

// NPMAX: row units a wave may compute one after the other
template <int RW, int NB, int NW, int NBUF, int U, int WPE, int NPMAX>
__global__ void __launch_bounds__(NW * 64, WPE) spconv_patch_kernel(ConvPatchArgs args)
{
    using Cfg = ConvPatchCfg<RW>;
    constexpr bool R16 = Cfg::R16;
    constexpr int NA = Cfg::NA, MBW = Cfg::MBW, STEPS = Cfg::STEPS;
    constexpr int NCB = R16 ? NB * 2 : NB;           // column blocks of a wave: 16 or 32 columns
    constexpr int AV = R16 ? 4 : 16;                 // accumulator values per lane and block
    constexpr int NQ = MBW * NCB * AV / 4;           // quads of accumulator values per lane
    constexpr bool WIDE = NPMAX > conv_patch_units(RW); // all filters in one workgroup
    // U: items of the patch a thread keeps in flight; WPE: waves per SIMD the registers are kept to
    constexpr int RING_OPS = NBUF * Cfg::OPS;
    static_assert(NBUF % 2 == 0 && NBUF <= CONV_PATCH_TAIL_BATCHES && RING_OPS + 2 < 64, "fragment sets alternate; vmcnt is a 6-bit counter");

    extern __shared__ __attribute__((aligned(1024))) char lds_raw[];
    const uint32_t lds0 = (uint32_t)(uintptr_t)(SHFLBW_LDS char*)lds_raw;
    // What the way to the first loads of the patch reads of the arguments is asked for at once: left to the compiler it is loaded where
    // it is used, a dozen trips to the scalar cache one after the other.
    ConvPatchArgs a = args;
    in_registers(a.p.jobs_per_xcd, a.p.jobs, a.p.chunks, a.p.magic_chunks, a.p.blocks_hw, a.p.magic_bhw, a.p.blocks_w, a.p.magic_bw,
                 a.p.units, a.p.tile_h, a.p.tile_w, a.p.stride, a.p.pad_h, a.p.pad_w, a.p.H, a.p.W, a.p.Ho, a.p.npos, a.p.pitch,
                 a.p.magic_pg, a.p.patch_w, a.p.magic_pw, a.p.skip, a.p.in_bytes, a.C, a.in, a.p.groups, a.p.kshift, a.p.panels_per_wave, a.F,
                 a.first_batch);
    const ConvPatchPlan& P = a.p;
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // XCD x owns a contiguous range of the jobs (column tile, chunk of filters), chunk-minor: the workgroups that write
    // interleaved filters of the same pixels share an L2, where their partial lines meet
    const int xcd = blockIdx.x & 7, job = xcd * P.jobs_per_xcd + (int)(blockIdx.x >> 3);
    if (job >= min(P.jobs, (xcd + 1) * P.jobs_per_xcd)) return;
    int tile, ch;
    fast_divmod(job, P.chunks, P.magic_chunks, tile, ch);

    // ---- this wave's row units (their batches of 32 slots lie one unit behind the other in memory); the trip to where they begin is
    // under way while the patch is asked for
    const int grp = wave >> P.kshift, np = P.panels_per_wave, nunits = a.F / RW;
    const int ufirst = (ch * P.groups + grp) * np;
    auto first_of = [&](int j) __attribute__((always_inline)) { // batch the wave's unit j begins with
        return ((const SHFLBW_CONST int*)(uintptr_t)a.first_batch)[min(ufirst + min(j, np), nunits)];
    };
    constexpr int NPB = WIDE ? 1 : NPMAX;
    int bound[NPB + 1]; // batches of unit j: [bound[j], bound[j + 1]); wide: those of all the wave's units
#pragma unroll
    for (int j = 0; j <= NPB; j++) bound[j] = first_of(WIDE ? j * NPMAX : j);
    // (wide: the ends of the unit computed and of the next one, a unit ahead of their use; all of them in an array would be an array in memory)
    int unit_end = 0, next_end = 0;
    if constexpr (WIDE) unit_end = first_of(1), next_end = first_of(2);

    // ---- the unit of this lane's column (lane % 4): its first output and input pixel.  A unit past the end lies outside.
    SHFLBW_LDS int* tout = (SHFLBW_LDS int*)(uintptr_t)lds0;
    const uint32_t slab = lds0 + 32 * NB * 4;
    int img, oh, ow; // of the lane's unit: image, first output row and column
    int uh[4], uw[4], ub[4];
    {
        const int unit = tile * 4 + (lane & 3);
        int rem, bi, bj;
        fast_divmod(unit, P.blocks_hw, P.magic_bhw, img, rem);
        fast_divmod(rem, P.blocks_w, P.magic_bw, bi, bj);
        const bool ok = unit < P.units;
        const int oh0 = bi * P.tile_h, h0 = oh0 * P.stride - P.pad_h;
        oh = ok ? oh0 : P.Ho, ow = bj * P.tile_w;
        const int h = ok ? h0 : P.H, w = ow * P.stride - P.pad_w;
        const int b = (int)((unsigned)((img * P.H + h) * P.W + w) * (unsigned)(a.C * 2));
#pragma unroll
        for (int u = 0; u < 4; u++) {
            uh[u] = __builtin_amdgcn_readlane(h, u);
            uw[u] = __builtin_amdgcn_readlane(w, u);
            ub[u] = __builtin_amdgcn_readlane(b, u);
        }
    }

    struct Batch {
        half8_t a[NA];
        typename std::conditional<R16, int, int2_t>::type i; // LDS offsets in units of 8 bytes, 16 bits each: slots s, s + 4 of every step
    };
    struct Frags {
        half8_t b[STEPS][NCB];
    };
    int ks, left, fpos, fend; // this wave's share of the batches
    // ---- every load up to the end of the products is inline assembly with hand-written waits: the patch, the places
    // and the ring of batches share one counter, and the compiler would wait for all of them at the first use of one
    const uint32_t lane16 = (uint32_t)lane * 16;
    const uint32_t offl = R16 ? (uint32_t)((lane >> 4) * 4 + (li >> 2)) * 4 : (uint32_t)((lane >> 5) * 4 + (li >> 2)) * 8;
    // Past the wave's last batch the loads are issued without a lane: no traffic, and the waits go on counting the same
    // number of them.
    auto fetch = [&](Batch& b) __attribute__((always_inline)) {
        const char* A = (const char*)a.packedA + (size_t)fpos * (32 * RW * 2);
        const char* I = (const char*)a.offs + (size_t)fpos * 64;
        if constexpr (NA == 4)
            asm volatile("s_cmp_lt_i32 %[p], %[e]\n\t"
                         "s_cselect_b64 exec, -1, 0\n\t"
                         "global_load_dwordx4 %[a0], %[l], %[A]\n\t"
                         "global_load_dwordx4 %[a1], %[l], %[A] offset:1024\n\t"
                         "global_load_dwordx4 %[a2], %[l], %[A] offset:2048\n\t"
                         "global_load_dwordx4 %[a3], %[l], %[A] offset:3072\n\t"
                         "global_load_dwordx2 %[i], %[o], %[I]\n\t"
                         "s_mov_b64 exec, -1"
                         : [a0] "=&v"(b.a[0]), [a1] "=&v"(b.a[1]), [a2] "=&v"(b.a[2]), [a3] "=&v"(b.a[3]), [i] "=&v"(b.i)
                         : [p] "s"(fpos), [e] "s"(fend), [l] "v"(lane16), [A] "s"(A), [o] "v"(offl), [I] "s"(I)
                         : "scc");
        else if constexpr (NA == 2)
            asm volatile("s_cmp_lt_i32 %[p], %[e]\n\t"
                         "s_cselect_b64 exec, -1, 0\n\t"
                         "global_load_dwordx4 %[a0], %[l], %[A]\n\t"
                         "global_load_dwordx4 %[a1], %[l], %[A] offset:1024\n\t"
                         "global_load_dwordx2 %[i], %[o], %[I]\n\t"
                         "s_mov_b64 exec, -1"
                         : [a0] "=&v"(b.a[0]), [a1] "=&v"(b.a[1]), [i] "=&v"(b.i)
                         : [p] "s"(fpos), [e] "s"(fend), [l] "v"(lane16), [A] "s"(A), [o] "v"(offl), [I] "s"(I)
                         : "scc");
        else
            asm volatile("s_cmp_lt_i32 %[p], %[e]\n\t"
                         "s_cselect_b64 exec, -1, 0\n\t"
                         "global_load_dwordx4 %[a0], %[l], %[A]\n\t"
                         "global_load_dword %[i], %[o], %[I]\n\t"
                         "s_mov_b64 exec, -1"
                         : [a0] "=&v"(b.a[0]), [i] "=&v"(b.i)
                         : [p] "s"(fpos), [e] "s"(fend), [l] "v"(lane16), [A] "s"(A), [o] "v"(offl), [I] "s"(I)
                         : "scc");
        fpos++;
    };
    auto pass_through = [](Batch& b) __attribute__((always_inline)) {
        asm volatile("" : "+v"(b.i));
#pragma unroll
        for (int q = 0; q < NA; q++) asm volatile("" : "+v"(b.a[q]));
    };
    // waits until at most `younger` batches fetched behind this one are outstanding
    auto arrived = [&](Batch& b, auto younger) __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(decltype(younger)::value * Cfg::OPS));
        pass_through(b);
    };
    Batch buf[NBUF];
    int touched0, touched1;

    auto share = [&]() __attribute__((always_inline)) {
        ks = wave & (P.ksplit - 1);
        if (!WIDE && (NPMAX == 1 || P.ksplit > 1)) {
            const int n = bound[1] - bound[0], b0 = bound[0];
            bound[0] = b0 + ((n * ks) >> P.kshift);
#pragma unroll
            for (int j = 1; j <= NPB; j++) bound[j] = b0 + ((n * (ks + 1)) >> P.kshift);
        }
        left = bound[NPB] - bound[0];
        fpos = bound[0];
        fend = bound[NPB];
    };
    int dst[NPMAX][MBW]; // places of this wave's rows in the staged output

    // ---- the patch: a lane takes 8 channels of one position in all four units (four 16-byte loads; bytes outside the
    // image come back as zeros from the bounds check of the buffer) and writes them as eight 8-byte pieces, one per
    // channel row.  The pitch is an odd multiple of 8 bytes: the 4 channel groups x 8 positions of half a wave fall into
    // different banks.
    {
        const int C8 = a.C >> 3, npos = P.npos, pitch = P.pitch, PG = (npos + 7) >> 3;
        const int combos = PG * ((C8 + 7) >> 3);
        const int ol = (lane & 3) | ((lane >> 5) << 2), pl = (lane >> 2) & 7;
        const int4_t rsrc = {(int)(uint32_t)(uintptr_t)a.in, (int)(uint32_t)((uintptr_t)a.in >> 32), (int)P.in_bytes, 0x00027000};
        half8_t v[U][4];
        uint32_t to[U];
        // Workgroups of eight waves ask for their first batches between the items of the patch, as these arrive: in front of them all,
        // the copies of the batches, 147 KB of a compute unit at 64 bytes a clock, held up the first write into LDS by 1.1 us.
        // Where the last round of a wave is not whole, items past the last one are not asked for and the first wait is for all of its
        // items: a load without a lane, which kept the counts of the waits the same, takes as long to issue as one with all of them
        // (32 x 28 x 28 x 128 -> 512, block height 32, 10 items for 8 waves: 21.0 us with such loads, 19.5 without).
        constexpr bool BETWEEN = NW == 8;
        auto load_round = [&](int q0) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < U; k++) {
                const int q = q0 + k * NW;
                to[k] = 0xffffffffu;
                uint32_t at[4] = {0, 0, 0, 0};
                if (q < combos) {
                    int og, pg, pi, pj;
                    fast_divmod(q, PG, P.magic_pg, og, pg);
                    const int oct = og * 8 + ol, pos = pg * 8 + pl;
                    fast_divmod(pos, P.patch_w, P.magic_pw, pi, pj);
                    if (P.skip) { // a stride wider than the filter: input rows and columns no tap reads are left out
                        if (P.stride > a.R) pi = (pi / a.R) * P.stride + pi % a.R;
                        if (P.stride > a.S) pj = (pj / a.S) * P.stride + pj % a.S;
                    }
                    const bool in_patch = oct < C8 && pos < npos;
                    to[k] = in_patch ? (uint32_t)(oct * 8) * pitch + pos * 8 : 0xffffffffu;
                    const uint32_t rel = (uint32_t)((pi * P.W + pj) * a.C + oct * 8) * 2;
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const bool ok = in_patch && (unsigned)(uh[u] + pi) < (unsigned)P.H && (unsigned)(uw[u] + pj) < (unsigned)P.W;
                        at[u] = ok ? rel + (uint32_t)ub[u] : 0xffffffffu;
                    }
                }
                if (q >= combos) continue;
                asm volatile("buffer_load_dwordx4 %[v0], %[a0], %[r], 0 offen\n\t"
                             "buffer_load_dwordx4 %[v1], %[a1], %[r], 0 offen\n\t"
                             "buffer_load_dwordx4 %[v2], %[a2], %[r], 0 offen\n\t"
                             "buffer_load_dwordx4 %[v3], %[a3], %[r], 0 offen"
                             : [v0] "=&v"(v[k][0]), [v1] "=&v"(v[k][1]), [v2] "=&v"(v[k][2]), [v3] "=&v"(v[k][3])
                             : [a0] "v"(at[0]), [a1] "v"(at[1]), [a2] "v"(at[2]), [a3] "v"(at[3]), [r] "s"(rsrc));
            }
        };
        auto write_item = [&](int k) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < 4; u++) asm volatile("" : "+v"(v[k][u]));
            if (to[k] != 0xffffffffu) {
                uint32_t at = slab + to[k];
                const int4_t d0 = __builtin_bit_cast(int4_t, v[k][0]), d1 = __builtin_bit_cast(int4_t, v[k][1]),
                             d2 = __builtin_bit_cast(int4_t, v[k][2]), d3 = __builtin_bit_cast(int4_t, v[k][3]);
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const unsigned sel = (e & 1) ? 0x07060302u : 0x05040100u;
                    int2_t w;
                    w.x = (int)__builtin_amdgcn_perm((unsigned)d1[e >> 1], (unsigned)d0[e >> 1], sel);
                    w.y = (int)__builtin_amdgcn_perm((unsigned)d3[e >> 1], (unsigned)d2[e >> 1], sel);
                    *(SHFLBW_LDS int2_t*)(uintptr_t)at = w;
                    at += pitch;
                }
            }
        };
        int q0 = wave;
        for (; q0 + NW * U < combos; q0 += NW * U) {
            load_round(q0);
            asm volatile("s_waitcnt vmcnt(0)");
#pragma unroll
            for (int k = 0; k < U; k++) write_item(k);
        }
        load_round(q0); // the last round, maybe empty for this wave
        const bool whole_round = q0 + NW * (U - 1) < combos;

        // ---- while it is on its way (the arguments anew: kept from the start they would not fit the scalar registers)
        const SHFLBW_CONST ConvPatchArgs* again = (const SHFLBW_CONST ConvPatchArgs*)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(again));
        a = *(const ConvPatchArgs*)again;
        in_registers(a.p.ksplit, a.p.kshift, a.F, a.packedA, a.offs, a.dst, a.p.touch_bytes, a.p.touch_step,
                     a.p.Wo, a.p.row_len, a.p.magic_row);
        share();
        // places of this wave's rows in the staged output
#pragma unroll
        for (int j = 0; j < NPMAX; j++)
#pragma unroll
            for (int mb = 0; mb < MBW; mb++) {
                const uint32_t at = (uint32_t)min((ufirst + j) * RW + mb * 32 + (lane & (R16 ? 15 : 31)), a.F - 1) * 2;
                asm volatile("global_load_ushort %0, %1, %2" : "=v"(dst[j][mb]) : "v"(at), "s"(a.dst));
            }
        if (tid < 32 * NB) { // output pixel of every column of the tile, -1: none
            int i, j;
            fast_divmod(tid >> 2, P.row_len, P.magic_row, i, j);
            tout[tid] = i < P.tile_h && j < P.tile_w && oh + i < P.Ho && ow + j < P.Wo ? (img * P.Ho + oh + i) * P.Wo + ow + j : -1;
        }
        constexpr int FPI = BETWEEN ? (NBUF + U - 1) / U : NBUF, PLACES = NPMAX * MBW;
        static_assert((U - 1) * 4 + PLACES + RING_OPS < 64, "vmcnt is a 6-bit counter");
        // The filter is not in the L2 when a launch starts, and the workgroups of an XCD walk it in step: left to the ring,
        // every batch would cost all of them a trip to memory.  Each thread touches a line of its own once, which brings
        // the whole image into the XCD's L2 while the patch is on its way.
        auto touch = [&]() __attribute__((always_inline)) {
            const uint32_t line = ((blockIdx.x >> 3) * (NW * 64) + tid) * 128;
            asm volatile("global_load_dword %0, %1, %2" : "=v"(touched0) : "v"(min(line, P.touch_bytes)), "s"(a.packedA));
            asm volatile("global_load_dword %0, %1, %2" : "=v"(touched1) : "v"(min(line + P.touch_step, P.touch_bytes)), "s"(a.packedA));
        };
        auto items = [&](auto self, auto kk) __attribute__((always_inline)) {
            constexpr int k = decltype(kk)::value, ahead = FPI * (k + 1) < NBUF ? FPI * (k + 1) : NBUF;
            if constexpr (k < U) {
#pragma unroll
                for (int j = FPI * k; j < ahead; j++) fetch(buf[j]);
                if (k == U - 1 || !whole_round)
                    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(ahead * Cfg::OPS));
                else
                    asm volatile("s_waitcnt vmcnt(%0)" : : "n"((U - 1 - k) * 4 + PLACES + ahead * Cfg::OPS));
                write_item(k);
                self(self, std::integral_constant<int, k + 1>{});
            }
        };
        if constexpr (BETWEEN) {
            items(items, std::integral_constant<int, 0>{});
            touch();
        } else { // (items past the last one were left out: one wait for all)
#pragma unroll
            for (int j = 0; j < NBUF; j++) fetch(buf[j]);
            touch();
            asm volatile("s_waitcnt vmcnt(%0)" : : "n"(RING_OPS + 2));
#pragma unroll
            for (int k = 0; k < U; k++) write_item(k);
        }
#pragma unroll
        for (int j = 0; j < NPMAX; j++)
#pragma unroll
            for (int mb = 0; mb < MBW; mb++) asm volatile("" : "+v"(dst[j][mb])); // older than the ring: arrived
        // the row of zeros the padding slots read, and behind it what columns without a pixel may touch
        for (int i = tid; i < (pitch + P.slack) >> 3; i += NW * 64)
            *(SHFLBW_LDS int2_t*)(uintptr_t)(slab + (uint32_t)a.C * pitch + i * 8) = int2_t{0, 0};
    }
    __syncthreads(); // the patch

    // ---- products
    uint32_t colc[NCB]; // LDS offset of the lane's four columns
#pragma unroll
    for (int nb = 0; nb < NCB; nb++) {
        const int pos = R16 ? nb * 4 + (li & 3) : nb * 8 + ((lane >> 4) & 1) * 4 + (li & 3);
        int i, j;
        fast_divmod(pos, P.row_len, P.magic_row, i, j);
        colc[nb] = slab + (i < P.tile_h ? (uint32_t)(i * P.step_h * P.patch_w + j * P.step_w) * 8 : 0u);
    }
    typedef float accv_t __attribute__((ext_vector_type(AV)));
    accv_t acc[MBW][NCB];
    constexpr int NKEPT = WIDE ? 1 : NPMAX;
    half4_t kept[NKEPT][NQ]; // finished panels, rounded to fp16
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int mb = 0; mb < MBW; mb++)
#pragma unroll
            for (int nb = 0; nb < NCB; nb++)
#pragma unroll
                for (int i = 0; i < AV; i++) acc[mb][nb][i] = 0.f;
    };
    clear();
#pragma unroll
    for (int j = 0; j < NKEPT; j++)
#pragma unroll
        for (int q = 0; q < NQ; q++) kept[j][q] = half4_t{0, 0, 0, 0};
    // The results' LDS rows: where the patch was; behind the patch in the wide kernels, whose units go there as they are finished
    const uint32_t SP = WIDE || a.dense ? NB * 64 + 16 : NB * 64 + 8;
    uint32_t stage = slab;
    if constexpr (WIDE) stage += ((uint32_t)(a.C + 1) * P.pitch + P.slack + 15) & ~15u;
    auto put = [&](const int(&place)[MBW], int q, half4_t h) __attribute__((always_inline)) { // quad q of the lane's values of a unit
        const int i = q * 4, mb = i / (NCB * AV), nb = (i / AV) % NCB, ig = (i % AV) / 4;
        const uint32_t col = R16 ? nb * 16 + (lane >> 4) * 4 : nb * 32 + ig * 8 + (lane >> 5) * 4;
        *(SHFLBW_LDS half4_t*)(uintptr_t)(stage + place[mb] * SP + col * 2) = h;
    };
    {
        auto read_frags = [&](const Batch& b, Frags& f) __attribute__((always_inline)) {
#pragma unroll
            for (int h = 0; h < STEPS; h++)
#pragma unroll
                for (int nb = 0; nb < NCB; nb++) {
                    uint32_t both;
                    if constexpr (R16) both = (uint32_t)b.i;
                    else both = (uint32_t)b.i[h];
                    const half4_t l = lds_read_tr16(((both & 0xffff) << 3) + colc[nb]);
                    const half4_t u = lds_read_tr16(((both >> 16) << 3) + colc[nb]);
                    f.b[h][nb] = __builtin_shufflevector(l, u, 0, 1, 2, 3, 4, 5, 6, 7);
                }
        };
        auto mma = [&](const Frags& f, const Batch& b) __attribute__((always_inline)) {
#pragma unroll
            for (int h = 0; h < STEPS; h++)
#pragma unroll
                for (int mb = 0; mb < MBW; mb++)
#pragma unroll
                    for (int nb = 0; nb < NCB; nb++) {
                        if constexpr (R16)
                            acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f.b[h][nb], b.a[0], acc[mb][nb], 0, 0, 0);
                        else
                            acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.b[h][nb], b.a[h * MBW + mb], acc[mb][nb], 0, 0, 0);
                    }
        };
        // end of a unit: its sums to fp16 (with a split over the kept columns a wave has one unit, whose fp32 sums stay
        // in acc), then the next unit that has batches
        int cur = 0, pos = bound[0], end = WIDE ? unit_end : bound[1];
        auto next_unit = [&]() __attribute__((always_inline)) {
            if constexpr (WIDE) {
#pragma unroll 1
                while (pos == end && cur < np && ufirst + cur < nunits) {
                    int place[MBW];
#pragma unroll
                    for (int mb = 0; mb < MBW; mb++) {
                        place[mb] = dst[0][mb];
#pragma unroll
                        for (int t = 1; t < NPMAX; t++) {
                            int of_t = dst[t][mb];
                            asm("" : "+v"(of_t)); // (a choice between values: from one between elements the compiler makes an array in memory)
                            place[mb] = t == cur ? of_t : place[mb];
                        }
                    }
#pragma unroll
                    for (int q = 0; q < NQ; q++) {
                        half4_t h;
#pragma unroll
                        for (int e = 0; e < 4; e++) h[e] = (half_t)acc[(q * 4 + e) / (NCB * AV)][((q * 4 + e) / AV) % NCB][(q * 4 + e) % AV];
                        put(place, q, h);
                    }
                    clear();
                    cur++;
                    end = next_end;
                    next_end = first_of(cur + 2);
                }
                return;
            }
#pragma unroll
            for (int j = 0; j < NKEPT; j++) // units without a batch in front are passed over
                if (cur < NPMAX && pos == end) {
                    if (P.ksplit > 1) { cur = NPMAX; break; }
#pragma unroll
                    for (int t = 0; t < NKEPT; t++)
                        if (t == cur) {
#pragma unroll
                            for (int q = 0; q < NQ; q++)
#pragma unroll
                                for (int e = 0; e < 4; e++) {
                                    const int i = q * 4 + e;
                                    kept[t][q][e] = (half_t)acc[i / (NCB * AV)][(i / AV) % NCB][i % AV];
                                }
                        }
                    clear();
                    cur++;
                    int e = bound[NPB];
#pragma unroll
                    for (int t = 0; t < NPB; t++) e = t == cur ? bound[t + 1] : e;
                    end = e;
                }
        };
        if constexpr (NPMAX > 1) next_unit();
        Frags fr[2];
        if (left > 0) {
            arrived(buf[0], std::integral_constant<int, NBUF - 1>{});
            read_frags(buf[0], fr[0]);
        }
        // MFMAs of a batch first, the LDS reads of the next one spread behind them
        auto interleave = [&]() __attribute__((always_inline)) {
            constexpr int NRD = STEPS * NCB * 2, NMM = STEPS * MBW * NCB, RPM = (NRD + NMM - 1) / NMM;
#pragma unroll
            for (int i = 0; i < NMM; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
                __builtin_amdgcn_sched_group_barrier(0x100, RPM, 0); // LDS reads
            }
        };
        for (; left > NBUF; left -= NBUF) {
#pragma unroll
            for (int j = 0; j < NBUF; j++) {
                arrived(buf[(j + 1) % NBUF], std::integral_constant<int, NBUF - 2>{});
                read_frags(buf[(j + 1) % NBUF], fr[(j + 1) & 1]);
                mma(fr[j & 1], buf[j]);
                interleave();
                fetch(buf[j]);
                if constexpr (NPMAX > 1)
                    if (++pos == end) next_unit();
            }
        }
        // the rest: what it needs is in the ring
        auto rest = [&](auto self, auto jj) __attribute__((always_inline)) {
            constexpr int j = decltype(jj)::value;
            if constexpr (j < NBUF) {
                if (j < left) {
                    if constexpr (j + 1 < NBUF)
                        if (j + 1 < left) {
                            arrived(buf[j + 1], std::integral_constant<int, NBUF - 2 - j>{});
                            read_frags(buf[j + 1], fr[(j + 1) & 1]);
                        }
                    mma(fr[j & 1], buf[j]);
                    if constexpr (NPMAX > 1)
                        if (++pos == end) next_unit();
                }
                self(self, std::integral_constant<int, j + 1>{});
            }
        };
        rest(rest, std::integral_constant<int, 0>{});
        // no load may land in a register that has found another use
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(touched0), "+v"(touched1));
#pragma unroll
        for (int j = 0; j < NBUF; j++) pass_through(buf[j]);
    }

    const int row0 = ch * P.rows_wg, rows = min(P.rows_wg, a.F - row0);

    // ---- results: one LDS row per filter, in output order (a lane holds four columns, the four units of a position, of
    // one filter per 8-byte write); the patch is no longer needed
    __syncthreads();
    if (!WIDE && P.ksplit > 1) { // sum the parts: every wave adds up its share of the quads of its group
        stage = slab + NW * NQ * 1024;
#pragma unroll
        for (int q = 0; q < NQ; q++) {
            float4_t v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = acc[(q * 4 + e) / (NCB * AV)][((q * 4 + e) / AV) % NCB][(q * 4 + e) % AV];
            *(SHFLBW_LDS float4_t*)(uintptr_t)(slab + (wave * NQ + q) * 1024 + lane * 16) = v;
        }
        __syncthreads();
    }
    if constexpr (WIDE) {
    } else if (P.ksplit > 1) {
        // (all parts asked for at once: read one after the other, each waited for the one before)
        auto sum = [&](auto parts) __attribute__((always_inline)) {
            constexpr int K = decltype(parts)::value, MINE = (NQ + K - 1) / K;
            float4_t v[MINE][K];
#pragma unroll
            for (int i = 0; i < MINE; i++) // quads ks, ks + K, ... of every part
#pragma unroll
                for (int k = 0; k < K; k++)
                    v[i][k] = *(SHFLBW_LDS float4_t*)(uintptr_t)(slab + ((grp * K + k) * NQ + min(ks + i * K, NQ - 1)) * 1024 + lane * 16);
#pragma unroll
            for (int i = 0; i < MINE; i++) {
                const int q = ks + i * K;
                float4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < K; k++)
#pragma unroll
                    for (int e = 0; e < 4; e++) s[e] += v[i][k][e];
                half4_t h;
#pragma unroll
                for (int e = 0; e < 4; e++) h[e] = (half_t)s[e];
                if (q < NQ) put(dst[0], q, h);
            }
        };
        if (ufirst < nunits) {
            if (NW == 8 && P.ksplit == 8)
                sum(std::integral_constant<int, 8>{});
            else if (P.ksplit == 4)
                sum(std::integral_constant<int, 4>{});
            else
                sum(std::integral_constant<int, 2>{});
        }
    } else {
#pragma unroll
        for (int j = 0; j < NPMAX; j++)
            if (j < np && ufirst + j < nunits) {
#pragma unroll
                for (int q = 0; q < NQ; q++) {
                    half4_t h = kept[j][q];
                    if constexpr (NPMAX == 1) {
#pragma unroll
                        for (int e = 0; e < 4; e++) h[e] = (half_t)acc[(q * 4 + e) / (NCB * AV)][((q * 4 + e) / AV) % NCB][(q * 4 + e) % AV];
                    }
                    put(dst[j], q, h);
                }
            }
    }
    if constexpr (!WIDE) __syncthreads();
    if (WIDE || a.dense) { // transposing reads: a lane gets 8 consecutive filters of one of 16 pixels, twice, 32 filters apart; lanes
                   // 8..15 of each 16 then trade places so that a store writes whole 128-byte lines of 8 pixels
        const int nit = NB * 2 * ((rows + 63) >> 6);
        auto whole_lines = [&](auto mode) __attribute__((always_inline)) {
            for (int it = wave; it < nit; it += NW) {
                const int cb = it & (NB * 2 - 1), r0 = (it / (NB * 2)) * 64, g8 = (lane >> 4) * 8;
                int4_t v[2];
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const uint32_t at = stage + (uint32_t)(min(r0 + h * 32 + g8, rows - 8) + (li >> 2)) * SP + cb * 32 + (li & 3) * 8;
                    const half4_t lo = lds_read_tr16(at), hi = lds_read_tr16(at + 4 * SP);
                    v[h] = __builtin_bit_cast(int4_t, (half8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                }
                int4_t first, second;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    first[e] = __builtin_amdgcn_update_dpp(v[0][e], v[1][e], 0x128, 0xf, 0xc, false);  // row_ror:8 into lanes 8..15
                    second[e] = __builtin_amdgcn_update_dpp(v[1][e], v[0][e], 0x128, 0xf, 0x3, false); // ... into lanes 0..7
                }
                const int r = r0 + g8 + (li >> 3) * 32;
                const int pix0 = tout[cb * 16 + (li & 7)], pix1 = tout[cb * 16 + 8 + (li & 7)];
                if (pix0 >= 0 && r < rows) store_result_16B<decltype(mode)::value>(a.out + (size_t)pix0 * a.F + row0 + r, __builtin_bit_cast(half8_t, first));
                if (pix1 >= 0 && r < rows) store_result_16B<decltype(mode)::value>(a.out + (size_t)pix1 * a.F + row0 + r, __builtin_bit_cast(half8_t, second));
            }
        };
        if (a.streams)
            whole_lines(std::integral_constant<StoreMode, STORE_STREAM>{});
        else
            whole_lines(std::integral_constant<StoreMode, STORE_THROUGH>{});
    } else { // a chunk's filters are scattered over the pixel: 2-byte pieces in ascending order, merged in the L2
        constexpr int MAXQ = 8;
        int f[MAXQ];
#pragma unroll
        for (int q = 0; q < MAXQ; q++) f[q] = q * 64 + lane < rows ? a.filt[row0 + q * 64 + lane] : -1;
        for (int pos = wave; pos < 8 * NB; pos += NW) {
            half_t* o[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int pix = __builtin_amdgcn_readfirstlane(tout[pos * 4 + u]);
                o[u] = pix >= 0 ? a.out + (size_t)pix * a.F : nullptr;
            }
#pragma unroll
            for (int q = 0; q < MAXQ; q++)
                if (f[q] >= 0) {
                    const half4_t v = *(SHFLBW_LDS half4_t*)(uintptr_t)(stage + (q * 64 + lane) * SP + pos * 8);
#pragma unroll
                    for (int u = 0; u < 4; u++)
                        if (o[u]) o[u][f[q]] = v[u];
                }
        }
    }
}

// One thread a lane's piece of a fragment: 8 slots of one row.  Once per filter image; neighbouring lanes read neighbouring rows
// of a kept vector.  (On the host, packing the 1.9 MB of a 2048 x 512 x 3 x 3 filter at density 0.1 takes 85 us and copying them 76.)
__global__ void __launch_bounds__(256) patch_pack_kernel(const half_t* values, const int* src, half8_t* packedA, int rows, size_t pieces)
{
    const size_t q = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= pieces) return;
    const int lane = (int)(q & 63), per_batch = rows == 16 ? 1 : rows / 16, blocks = rows / 32;
    const size_t batch = (q >> 6) / per_batch;
    const int frag = (int)((q >> 6) - batch * per_batch);
    const int row = rows == 16 ? lane & 15 : frag % blocks * 32 + (lane & 31);
    const int slot = rows == 16 ? (lane >> 4) * 8 : frag / blocks * 16 + (lane >> 5) * 8;
    half8_t v;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int from = src[batch * 32 + slot + j];
        v[j] = from < 0 ? (half_t)0 : values[(size_t)from * rows + row];
    }
    packedA[q] = v;
}

hipError_t launch_patch_pack(const half_t* values, const int* src, half8_t* packedA, int rows, size_t batches, hipStream_t stream)
{
    const size_t pieces = batches * rows * 4; // 32 slots of `rows` values, 8 a piece
    if (pieces == 0) return hipSuccess;
    if ((pieces + 255) / 256 * 256 > 0xffffffffull) return hipErrorInvalidValue;
    hipLaunchKernelGGL(patch_pack_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, stream, values, src, packedA, rows, pieces);
    return hipGetLastError();
}

template <int RW, int NB, int NW, int NBUF, int U, int WPE, int NPMAX>
static hipError_t launch_patch(const ConvPatchArgs& a, hipStream_t stream)
{
    hipLaunchKernelGGL((spconv_patch_kernel<RW, NB, NW, NBUF, U, WPE, NPMAX>), dim3(a.p.jobs_per_xcd * 8), dim3(NW * 64), a.p.lds_bytes, stream, a);
    return hipGetLastError();
}

template <int RW, int NB, int NW, int NBUF, int U, int WPE, int NPMAX>
static hipError_t prepare_patch()
{
    return hipFuncSetAttribute((const void*)spconv_patch_kernel<RW, NB, NW, NBUF, U, WPE, NPMAX>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               CONV_PATCH_LDS_MAX);
}

#define SHFLBW_PATCH_UNITS(RW, NB, NW, NBUF, U, WPE, KIND, NPMAX) \
    {RW, NB, NW, KIND, WPE * 4 / NW, NBUF, U, NPMAX, &launch_patch<RW, NB, NW, NBUF, U, WPE, NPMAX>, &prepare_patch<RW, NB, NW, NBUF, U, WPE, NPMAX>}
#define SHFLBW_PATCH(RW, NB, NW, NBUF, U, WPE, DEEP) SHFLBW_PATCH_UNITS(RW, NB, NW, NBUF, U, WPE, DEEP, conv_patch_units(RW))

// Workgroups of four waves keep two batches in flight: a deeper ring is more code to fetch at the start of every launch (24 x 24 x 24 x
// 56 -> 32, 3 x 3, stride 2: 3.9 us, 4.4 with six batches), which only waves with many batches win back: for those the planner weighs
// its cuts with the deep kernels.  us, before / now: 2 x 44 x 44 x 136 -> 96, 3 x 3, block height 32 6.5 / 5.1, 16 x 50 x 50 x 160 -> 256, 1 x 7,
// 27.4 / 25.6, 3 x 14 x 30 x 224 -> 800, stride 2 6.8 / 6.1; block height 16: 8 x 26 x 52 x 48 -> 1216, stride 2 13.1 / 10.9, 8 x 45 x 41 x 24 -> 160
// 9.0 / 7.5.  As many batches as the registers of the cut's workgroups hold without spilling; row units of 64, and of 16 over 64
// columns, leave no room for them.
//
// Wide kernels (the last ones): a permuted filter of more rows than the waves of a workgroup otherwise compute leaves in 2-byte stores from
// every workgroup of a column tile, and what bounds those is the L2s' writes: 64 lanes of one of six workgroups reach thirteen pieces of 64
// bytes (17 x 18 x 14 x 208 -> 1472, 1 x 1: 4.9 of a workgroup's 8.4 us).  With up to four times the row units a wave, over 32 columns, or
// twice over 64, one workgroup has all filters of its pixels and stores whole lines.  A unit's results go to LDS behind the patch as the
// unit is finished: held in registers as in the other kernels they would not fit beside the ring.  us, in chunks / wide: that layer 12.6 /
// 9.3, 88 x 8 x 23 x 216 -> 1344, 3 x 3, block height 64 43.1 / 25.2, 43 x 13 x 27 x 824 -> 1184, 1 x 1, 32 38.4 / 24.5, 120 x 14 x 25 x 80
// -> 608, 1 x 1, 16 32.3 / 24.3, 16 x 33 x 33 x 192 -> 1536, 1 x 7, 128 55.0 / 45.8; 64 columns: 24 x 13 x 25 x 176 -> 832, 1 x 7, 32 21.5
// / 12.6 (19.5 over 32 columns), 8 x 54 x 54 x 240 -> 640, 3 x 3, 64 31.6 (41.2); sampled layers: see the estimate.  Layers of few pixels,
// which would leave compute units idle, stay in chunks, and so do filters of 2048 rows: a row of a result takes 80 bytes of LDS, which
// leaves no room for a patch.
static const ConvPatchKernel g_patch[] = {
    SHFLBW_PATCH(16, 2, 8, 8, 5, 2, 0), SHFLBW_PATCH(32, 2, 8, 8, 5, 2, 0), SHFLBW_PATCH(64, 2, 8, 4, 5, 2, 0),
    SHFLBW_PATCH(16, 1, 8, 8, 5, 2, 0), SHFLBW_PATCH(32, 1, 8, 8, 5, 2, 0), SHFLBW_PATCH(64, 1, 8, 4, 5, 2, 0),
    SHFLBW_PATCH(16, 2, 4, 2, 2, 3, 0), SHFLBW_PATCH(32, 2, 4, 2, 2, 2, 0), SHFLBW_PATCH(64, 2, 4, 2, 2, 3, 0),
    SHFLBW_PATCH(16, 1, 4, 2, 2, 4, 0), SHFLBW_PATCH(32, 1, 4, 2, 2, 4, 0), SHFLBW_PATCH(64, 1, 4, 2, 2, 4, 0),
    SHFLBW_PATCH(32, 2, 4, 6, 2, 2, 1), SHFLBW_PATCH(16, 1, 4, 6, 2, 4, 1), SHFLBW_PATCH(32, 1, 4, 4, 2, 4, 1),
    SHFLBW_PATCH_UNITS(16, 1, 8, 4, 5, 2, CONV_PATCH_WIDE, 16), SHFLBW_PATCH_UNITS(32, 1, 8, 4, 5, 2, CONV_PATCH_WIDE, 8),
    SHFLBW_PATCH_UNITS(16, 2, 8, 4, 5, 2, CONV_PATCH_WIDE, 8), SHFLBW_PATCH_UNITS(32, 2, 8, 4, 5, 2, CONV_PATCH_WIDE, 4),
    SHFLBW_PATCH_UNITS(64, 2, 8, 4, 5, 2, CONV_PATCH_WIDE, 2),
    SHFLBW_PATCH_UNITS(64, 1, 8, 4, 5, 2, CONV_PATCH_WIDE, 4),
};
static int patch_deep_batches(int rows) { return rows == 16 ? 13 : 9; } // of a wave, from which on the deeper ring is taken

// Estimated microseconds of the plane forms (three launches): the launches, the gathers of the SpMM, the two layout
// passes.  The weights come from a fit to 124 measured layers (20 % rms).
static double conv_planes_estimate(const ConvPatchProblem& q)
{
    const int s = q.stride;
    const double PW = q.Wo + (q.S - 1) / s, PH = q.Ho + (q.R - 1) / s, n = (double)q.B * q.Ho * PW;
    const double kept = (q.kept_per_panel + 32) * (q.F / q.V);
    const double in = 2.0 * q.B * q.H * q.W * q.C, planes = 2.0 * s * s * q.C * PH * PW * q.B, out = 2.0 * q.F * (n + (double)q.B * q.Ho * q.Wo);
    return 12.0 + kept * n * 2 / 15.1e6 + (in + planes) / 9.2e6 + out / 4.65e6;
}

ConvPatchShape conv_patch_shape(int rows, const ConvPatchPlan& p)
{
    ConvPatchShape shape{p.pitch, p.patch_w, 0};
    for (int t = 0; t < 32 / conv_patch_group(rows); t++) {
        const int i = t / p.row_len, j = t % p.row_len;
        if (i < p.tile_h) shape.foot |= 1u << ((i * p.step_h * p.patch_w + j * p.step_w) & 31);
    }
    return shape;
}

// The cut with the least estimated time: rounds of workgroups times the sum of a workgroup's phases.  The weights come from
// a fit to 124 layers measured with 20 to 40 cuts each (10 % rms; the cut it picks is 4 % slower than the best one
// measured on average).  Where the plane forms are estimated faster - many filters over few resident pixels (wide
// filters over many channels), filters of several workgroups interleaved in the output - the cut is not `preferred`:
// 7 x 54 x 54 x 584 -> 1024, 5 x 5, stride 2 takes 152 us here, 54 us there; 16 x 14 x 14 x 512 -> 2048, which it takes, 20 and 23 us.
// On 64 sampled layers it is preferred for 60, where the plane forms take 1.2 to 4.0 times as long.
bool conv_patch_plan(const ConvPatchProblem& q, ConvPatchPlan* plan, const std::vector<ConvPatchShape>* held, bool wide_cuts)
{
    ConvPatchPlan best{};
    double best_cost = 0, best_plain = 0, best_other = HUGE_VAL; // best_other: of the cuts that are not wide
    const bool flat = q.R == 1 && q.S == 1 && q.stride == 1; // every pixel for itself: one long row
    const unsigned long long in_bytes = (unsigned long long)q.B * q.H * q.W * q.C * 2;
    if (in_bytes > 0xffffff00ull || (unsigned long long)q.B * q.Ho * q.Wo > 0x7fffffffull) return false;
    const int B = flat ? 1 : q.B, H = flat ? 1 : q.H, W = flat ? q.B * q.H * q.W : q.W;
    const int Ho = flat ? 1 : q.Ho, Wo = flat ? W : q.Wo;
    const int eh = std::min(q.stride, q.R), ew = std::min(q.stride, q.S);
    const int rw = conv_patch_unit_rows(q.V), nunits = q.F / rw;
    const double batches = std::max(1.0, std::ceil(q.kept_per_panel / 32.0));
    for (const ConvPatchKernel& k : g_patch) {
        if (k.RW != rw) continue;
        const bool wide = k.deep == CONV_PATCH_WIDE;
        const int np_wide = (nunits + k.waves - 1) / k.waves; // row units of a wave with all filters in one workgroup
        if (wide && (!wide_cuts || !q.permuted || np_wide <= conv_patch_units(rw) || np_wide > k.units)) continue;
        const int positions = 8 * k.col_blocks;
        for (int th = 1; th <= std::min(positions, Ho); th++)
            for (int tw = 1; tw <= std::min(positions / th, Wo); tw++) {
                // rows of 8 or 16 positions: the 8 positions half a wave reads lie in a row (what the order of the slots counts
                // on); else positions are packed
                const int rl = tw <= 8 && th <= positions / 8 ? 8 : th == 1 ? 16 : tw;
                ConvPatchPlan p{};
                p.col_blocks = k.col_blocks, p.waves = k.waves, p.deep = k.deep;
                p.tile_h = th, p.tile_w = tw, p.row_len = rl;
                p.blocks_w = (Wo + tw - 1) / tw;
                const long blocks_hw = (long)((Ho + th - 1) / th) * p.blocks_w, units = B * blocks_hw;
                if (units > 0x3fffffffL) continue;
                p.blocks_hw = (int)blocks_hw;
                p.units = (int)units;
                const long tiles = (units + 3) / 4;
                p.patch_w = (tw - 1) * ew + q.S;
                p.npos = ((th - 1) * eh + q.R) * p.patch_w;
                p.pitch = 8 * (p.npos | 1);
                p.step_h = eh, p.step_w = ew;
                if (held && std::find(held->begin(), held->end(), conv_patch_shape(rw, p)) == held->end()) continue;
                // the furthest byte a lane reads: the last tap of the last channel, or the row of zeros, under the last
                // position of a row (positions from tile_w on are no pixels, but are read)
                const long last_row = std::max((long)q.C * p.pitch, (q.C - 1L) * p.pitch + ((q.R - 1L) * p.patch_w + q.S - 1) * 8);
                const long last = last_row + ((th - 1L) * eh * p.patch_w + (rl - 1L) * ew) * 8 + 8;
                p.slack = (int)std::max<long>(CONV_PATCH_SLACK, last - (q.C + 1L) * p.pitch);
                const long slab = (long)(q.C + 1) * p.pitch + p.slack;
                if (slab > CONV_PATCH_LDS_MAX) continue;
                // what the patch of a single workgroup takes, for a wide cut by its weight: a cut cannot be better than that
                const double rounds_patch = std::ceil((double)((p.npos + 7) / 8 * ((q.C + 63) / 64)) / (k.waves * k.items));
                const double start = 1.0 + (k.waves == 8 ? 1.15 : 0), patch_bytes = q.C * p.npos * 8 * 5.3e-6;
                if (best.valid && 2.9 + (start + patch_bytes + rounds_patch * 0.7) * (wide ? 0.65 : 1) >= best_cost) continue;
                for (int groups = k.waves; groups >= (wide ? k.waves : 1); groups >>= 1)
                    for (int np = wide ? np_wide : 1; np <= k.units; np = wide ? k.units + 1 : np << 1) {
                        p.groups = groups, p.ksplit = k.waves / groups, p.panels_per_wave = np;
                        if (p.ksplit > 1 && np > 1) continue;
                        if (groups > 1 && groups * np >= 2 * nunits) continue; // half of the waves would idle
                        for (p.kshift = 0; (1 << p.kshift) < p.ksplit; p.kshift++) {}
                        p.rows_wg = groups * np * rw;
                        p.chunks = (q.F + p.rows_wg - 1) / p.rows_wg;
                        const long jobs = tiles * p.chunks;
                        if (jobs > 0x3fffffffL) continue;
                        p.jobs = (int)jobs, p.jobs_per_xcd = (p.jobs + 7) / 8;
                        const int cols = 32 * k.col_blocks;
                        const long quads = (long)rw * cols / 64 / 4;
                        const long stage = (long)(wide ? q.F : p.rows_wg) * (cols * 2 + 16) + (p.ksplit > 1 ? k.waves * quads * 1024 : 0);
                        const long lds = 128 * k.col_blocks + (wide ? (slab + 15) / 16 * 16 + stage : std::max(slab, stage));
                        if (lds > CONV_PATCH_LDS_MAX) continue;
                        p.lds_bytes = (int)lds;
                        // ---- estimated microseconds
                        const int wgs = (int)std::min<long>(CONV_PATCH_LDS_MAX / lds, k.per_cu);
                        const double per_cu = std::ceil((double)jobs / q.cus), act = std::min<double>(wgs, per_cu);
                        const double rounds = std::ceil((double)jobs / ((double)q.cus * wgs));
                        const double w = k.waves * act; // waves of a compute unit
                        const double nb = std::ceil(np * batches / p.ksplit);
                        if (!wide && k.deep != (nb >= patch_deep_batches(rw) && conv_patch_kernel(rw, k.col_blocks, k.waves, 1) != nullptr)) continue;
                        const int steps = rw == 16 ? 1 : 2, mbw = rw == 64 ? 2 : 1, ncb = rw == 16 ? 2 * k.col_blocks : k.col_blocks;
                        const bool apart = rl == 8 || rl == 16; // rows of half a wave's positions lie in a line
                        const double t_mfma = steps * mbw * ncb * (rw == 16 ? 16 : 32) * w / 4 * 0.00045;
                        const double t_stream = w * (steps * mbw * 1024 + (rw == 16 ? 256 : 512)) / 64 * 0.0004;
                        const double t_lds = w * steps * ncb * 4 * (apart ? 1.2 : 2.0) * 0.00081;
                        const double t_longest = std::max(std::max(t_mfma, t_stream), std::max(t_lds, 0.37 / k.ring));
                        const double t_main = nb * (t_longest + 0.2 * (t_mfma + t_stream + t_lds - std::min(t_longest, t_mfma + t_stream + t_lds)));
                        const double t_patch = act * patch_bytes + rounds_patch * 0.7;
                        const double values = (double)cols * std::min(p.rows_wg, q.F) * act;
                        const double t_out = values * (!q.permuted || p.chunks == 1 ? 5.0e-5 : 1.5e-4) +
                                             (p.ksplit > 1 ? k.waves * rw * cols * 4.0 * act * 1.0e-5 : 0);
                        const double plain = start + t_patch + t_main + t_out;
                        // What surrounds the products costs the wide kernels less than this sum says, with the weights below by sampled
                        // layers near the line (0.65 alone: two of 42 that switch, of many products, 1.05 and 1.14 times as long; 0.55
                        // and 1.2: three 1.07 to 1.14); and a tie of the estimates goes to the chunks: 263 of 550 layers switch, 0.33 to 1.03
                        // times the time, 0.77 on average, two of them more than 1.02 (without the hundredth 280, ten of them up to 1.23:
                        // small layers of 576 filters, 9 x 46 x 5 x 144, 1 x 1 5.2 us, 6.4 on a wide cut).
                        const double one = wide ? std::min(plain, (start + t_patch + t_out) * 0.65 + t_main * 1.25) : plain;
                        const double cost = (2.9 + one * (1 + (rounds - 1) * 1.16) + jobs * 1.0e-5) * (wide ? 1.01 : 1);
                        if (!best.valid || cost < best_cost) {
                            best = p, best_cost = cost;
                            best_plain = 2.9 + plain * (1 + (rounds - 1) * 1.16) + jobs * 1.0e-5;
                            if (!wide) best_other = cost; // (the wide kernels come last: they do not stand in the way of another cut)
                            best.valid = 1;
                        }
                    }
            }
    }
    if (!best.valid) return false;
    // Without the wide kernels' weights, which were fitted against chunks (52 x 16 x 16 x 792 -> 1792, 1 x 1: 40.9 us here, 36.0 there); but a
    // layer that the form would take in chunks is not lost to the plane forms because a wide cut is estimated faster still.  Of 39450
    // sampled layers 9 are such; on these and five more the wide cut takes 0.47 to 0.99 times the plane forms' time and 0.77 to
    // 1.07 times that of the chunks: 23 x 38 x 38 x 168 -> 1984, 1 x 1, block height 64 77.9 us, planes 101.7, chunks 90.1.
    best.preferred = std::min(best_plain, best_other) <= conv_planes_estimate(q);
    best.H = H, best.W = W, best.Ho = Ho, best.Wo = Wo, best.stride = q.stride;
    best.pad_h = q.R / 2, best.pad_w = q.S / 2;
    best.skip = q.stride > q.R || q.stride > q.S;
    best.in_bytes = (unsigned)in_bytes;
    best.touch_bytes = best.touch_step = 0; // set with the size of the image
    best.magic_bhw = udiv_magic(best.blocks_hw);
    best.magic_bw = udiv_magic(best.blocks_w);
    best.magic_pw = udiv_magic(best.patch_w);
    best.magic_row = udiv_magic(best.row_len);
    best.magic_chunks = udiv_magic(best.chunks);
    best.magic_pg = udiv_magic((best.npos + 7) / 8);
    *plan = best;
    return true;
}

// Order of the kept columns of one row panel: the rows one pass of a transposing LDS read touches (32 lanes: four rows
// of 8 positions, for row units of 16 eight rows of 4) should fall into different banks.  A row starts in one of 32
// bank pairs; `foot` marks the pairs its positions touch when it starts in pair 0.  Exact tilings of the 32 pairs by
// shifted copies of `foot` are looked for first; groups are then filled from the tiling and shift whose
// scarcest member has the most rows left, and from whatever collides least once no tiling can be filled.
// It runs in the first initialisation of a layer, over every kept column: sets of bank pairs are words, so that a step
// does not walk the 32 pairs (14700 columns: 0.60 ms pair by pair, 0.10 ms so, on one machine).
static uint32_t rotated(uint32_t set, int by) { return by ? (set << by) | (set >> (32 - by)) : set; } // moved up by `by` pairs

// the starts from which a copy of the foot touches `set`
uint32_t ConvPatchOrder::touching(uint32_t set) const
{
    uint32_t starts = 0;
    for (uint32_t f = foot; f; f &= f - 1) starts |= rotated(set, (32 - __builtin_ctz(f)) & 31);
    return starts;
}

void ConvPatchOrder::find_tilings(std::vector<int>& shifts, uint32_t used)
{
    if ((int)shifts.size() == group) {
        tilings.push_back(shifts);
        return;
    }
    const uint32_t lowest = ~used & (used + 1); // the first pair without a row: some copy has to cover it
    for (uint32_t free = touching(lowest) & ~touching(used) & ~1u; free && tilings.size() < 3; free &= free - 1) {
        const int s = __builtin_ctz(free);
        shifts.push_back(s);
        find_tilings(shifts, used | rotated(foot, s));
        shifts.pop_back();
    }
}

ConvPatchOrder::ConvPatchOrder(uint32_t foot_, int group_) : foot(foot_), group(group_)
{
    std::vector<int> shifts{0};
    find_tilings(shifts, foot);
}

void ConvPatchOrder::of(const std::vector<int>& pair_of, std::vector<int>& order) const
{
    const int n = (int)pair_of.size();
    order.resize(n);
    int* out = order.data();
    const int* const end = out + n;
    int begin[33] = {}, count[32] = {}; // rows by start pair: by_pair[begin[s] ..], count[s] of them left
    for (int i = 0; i < n; i++) count[pair_of[i]]++;
    for (int s = 0; s < 32; s++) begin[s + 1] = begin[s] + count[s];
    std::vector<int> by_pair(n);
    int fill[32];
    std::copy(begin, begin + 32, fill);
    for (int i = 0; i < n; i++) by_pair[fill[pair_of[i]]++] = i;
    // left[c]: the pairs with at least c rows left
    std::vector<uint32_t> left(*std::max_element(count, count + 32) + 1, 0);
    for (int s = 0; s < 32; s++)
        for (int c = 0; c <= count[s]; c++) left[c] |= 1u << s;
    auto take = [&](int s) {
        *out++ = by_pair[begin[s + 1] - count[s]];
        left[count[s]--] &= ~(1u << s);
    };
    for (int c = (int)left.size() - 1; c > 0;) {
        uint32_t shifts = 0; // ... at which every member of a tiling has c rows left
        const std::vector<int>* with = nullptr;
        for (size_t t = 0; t < tilings.size() && !shifts; t++) {
            with = &tilings[t];
            shifts = ~0u;
            for (int d : tilings[t]) shifts &= rotated(left[c], (32 - d) & 31);
        }
        if (!shifts) {
            c--;
            continue;
        }
        for (int i = 0; i < c; i++)
            for (int d : *with) take((__builtin_ctz(shifts) + d) & 31);
    }
    const uint32_t meets = touching(foot); // the starts of rows that meet the row from pair 0
    int most = (int)left.size() - 1;
    while (out < end) {
        uint32_t level[9] = {}; // level[m]: pairs at least m of the picked rows touch
        uint32_t meeting = 0;   // the starts of rows that meet a picked one
        for (int g = 0; g < group && out < end; g++) {
            uint32_t from = left[1] & ~meeting;
            for (int m = 2; !from; m++) from = m <= g ? left[1] & ~touching(level[m]) : left[1];
            while (!left[most]) most--;
            int c = most; // of these the start with the most rows left, the lowest of equals
            while (!(left[c] & from)) c--;
            const int pick = __builtin_ctz(left[c] & from);
            const uint32_t row = rotated(foot, pick);
            for (int m = group; m > 1; m--) level[m] |= level[m - 1] & row;
            level[1] |= row;
            meeting |= rotated(meets, pick);
            take(pick);
        }
    }
}

const ConvPatchKernel* conv_patch_kernel(int rows, int col_blocks, int waves, int deep)
{
    for (const ConvPatchKernel& k : g_patch)
        if (k.RW == rows && k.col_blocks == col_blocks && k.waves == waves && k.deep == deep) return &k;
    return nullptr;
}

} // namespace shflbw
