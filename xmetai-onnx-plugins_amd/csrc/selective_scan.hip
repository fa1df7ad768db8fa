// SelectiveScanFn forward for gfx950 (CDNA4, wave64).
//
// Computes output 0 of the reference operator (selective_scan_fwd_kernel.cuh:
// 70-306): per channel (b,d) and state n,
//     delta' = softplus?(delta + bias),  h_t = exp2(delta'_t * A[d,n] * log2e) h_{t-1} + B_t delta'_t u_t,
//     y_t = D u_t + sum_n C_t h_t.
//
// Layout of the work (MI355X-first, not the reference's block scan):
//  * A lane owns SPL consecutive states of one channel and runs their
//    recurrences sequentially over the whole sequence, so every (t,n) costs
//    exactly one exp2 and four VALU ops; there is no cross-lane scan.
//  * LPC = ceil(N/SPL) lanes share a channel; a 256-thread workgroup owns
//    CPW = 256/LPC channels of one (batch, group), which share the B/C rows.
//  * The sequence is processed in tiles of 32 tokens.  Per tile the
//    workgroup loads u/delta rows and the B/C rows with coalesced 16-byte
//    loads (prefetched one tile ahead into registers), applies bias and
//    softplus once per (channel, token), and stages delta' and delta'*u in LDS.
//  * The LPC partial sums over states are added across lanes with DPP; one
//    lane per channel writes them to LDS and the store phase adds D*u and
//    writes y with 16-byte stores.
//  * z is never read: output 0 does not depend on it (reference
//    selective_scan_fwd_kernel.cuh:280 vs :296-299).
//  * The data tensors (u, delta, variable B/C, y) are fp32, or float16 /
//    bfloat16 as in the reference's half and bfloat16 instantiations
//    (input_t; A, D, bias, constant B/C are weight_t = fp32): loads convert
//    to fp32, the arithmetic is fp32, y is rounded to nearest even.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <type_traits>

#include "xm_hip.h"
#include "xm_params.h"
#include "selective_scan_dev.h"

namespace xm {
namespace {

using namespace ssdev;

constexpr int kThreads = 256;
// The kernel's part of the work (described at the kernel).
enum Mode { kWhole, kSegState, kSegOut };
struct SegSplit {
    int count, len;   // segments, tokens per segment (the last may be shorter)
};
// Sequence-split selection (ChoosePlan): considered below this many channel
// blocks (workgroups of the whole pass), for sequences at least this long.
constexpr long long kSegMaxChannelBlocks = 256;
constexpr int kSegMinSeqlen = 256;
constexpr long long kSplitMaxChannelBlocks = 320;
// Segments: enough workgroups for five per CU (what the VGPRs admit), of 128
// tokens or more.
constexpr long long kSplitTarget = 1280;
constexpr int kSplitMax = 16;
constexpr int kSplitMinLen = 128;

// Tokens per tile: 32 fp32 = one 128-byte line per (channel, tile), so every
// line of u and delta is consumed by the load that fetched it (rows are
// seqlen*4 bytes apart, a power of two at the benchmark shapes, and the other
// half of a line does not survive in L2 until the next tile).  256 channels
// per workgroup, or 128+ states, fall back to 16 tokens to stay within 64 KiB
// of LDS.
template <int CPW, int NP>
struct Tile {
    static constexpr int T = (CPW >= 256 || NP >= 128) ? 16 : 32;   // tokens per tile
    static constexpr int ROW = T + 4;                 // LDS row stride (padding breaks bank aliasing)
    static constexpr int Q4 = T / 4;                  // float4 groups per tile row
};

// Sum over the LPC consecutive lanes that share a channel (lane = c*LPC + q),
// result in all of them: xor 1 and 2 (quad_perm), xor 7 within 8 lanes
// (row_half_mirror), xor 8 (row_ror:8).
template <int LPC>
__device__ __forceinline__ float LaneGroupSum(float x) {
    if constexpr (LPC >= 2) x += DppF<0xB1>(x);
    if constexpr (LPC >= 4) x += DppF<0x4E>(x);
    if constexpr (LPC >= 8) x += DppF<0x141>(x);
    if constexpr (LPC >= 16) x += DppF<0x128>(x);
    return x;
}

// FAST: rows on 4-byte boundaries, dim_per_group % CPW == 0 and a workgroup's
// rows under 2 GiB.
// Full tiles then move as float4 with no guards, and the one-tile-ahead
// prefetch of u/delta/B/C stays in flight through the recurrence.  A ragged
// last tile (seqlen % 32 != 0) is peeled off the loop and loaded with guards.
// Without FAST every load is guarded (clamped address + select).
//
// MODE kWhole: the whole sequence.  The sequence split runs two launches of
// split.count segments of split.len tokens (a multiple of the tile) per
// channel block, so that few channel blocks still fill the chip:
//  * kSegState: segments 0 .. count - 2 from a zero state, the state alone (no
//    C, no y): 5.4 of the 8.2 issue slots per state and token of a whole
//    pass.  Writes each channel's sum of delta' and end state.
//  * kSegOut: every segment from its true start state, the composition of the
//    records of the segments before it (h <- exp2(A sum delta') h + h_end).  An
//    infinite state, whose decay over a segment may be 0 where no token's is,
//    would not be the whole pass's: the workgroup then walks the sequence from
//    its first token and stores only the segment's y.
// The records live in the output rows that the later segments will write:
// segment s's go into slot s of every later segment's rows, so a workgroup of
// the second launch reads only rows that it alone overwrites, before its
// first store, and no scratch is needed.
template <typename IT, int LPC, int SPL, bool BVAR, bool CVAR, bool FAST, int MODE>
__global__ __launch_bounds__(kThreads) void SelectiveScanFwdKernel(SelectiveScanParams p, SegSplit split) {
    constexpr int CPW = kThreads / LPC;      // channels per workgroup
    constexpr int NP = LPC * SPL;            // padded state count
    constexpr int kTile = Tile<CPW, NP>::T;
    constexpr int kRow = Tile<CPW, NP>::ROW;
    constexpr int kQ4 = Tile<CPW, NP>::Q4;
    constexpr int ITEMS = CPW * kQ4;         // (channel, 4-token) items per tile
    constexpr int IPT = (ITEMS + kThreads - 1) / kThreads;
    constexpr bool kState = MODE == kSegState;
    constexpr bool CLOAD = CVAR && !kState;   // C rows are read
    constexpr int NBC = (BVAR ? 1 : 0) + (CLOAD ? 1 : 0);
    constexpr int BCPT = NBC == 0 ? 1 : (NBC * NP * kQ4 + kThreads - 1) / kThreads;

    __shared__ __attribute__((aligned(16))) float sDl[CPW * kRow];        // delta' per (channel, token)
    __shared__ __attribute__((aligned(16))) float sDu[CPW * kRow];        // delta' * u
    __shared__ __attribute__((aligned(16))) float sB[BVAR ? NP * kRow : 1];
    __shared__ __attribute__((aligned(16))) float sC[CLOAD ? NP * kRow : 1];
    __shared__ __attribute__((aligned(16))) float sY[kState ? 1 : CPW * kRow];   // sum over states per (channel, token)

    const int tid = threadIdx.x;
    const int L = p.seqlen;
    const int N = p.dstate;
    const int dpg = p.dim_per_group;
    const int ncb = (dpg + CPW - 1) / CPW;
    int wg = blockIdx.x;
    int seg = 0, tb = 0, te = L;             // this workgroup's segment, its tokens [tb, te)
    if constexpr (MODE != kWhole) {
        const int blocks = ncb * p.groups_b * p.batch;
        seg = wg / blocks;
        wg -= seg * blocks;
        tb = seg * split.len;
        te = min(L, tb + split.len);
    }
    const int y_from = tb;                   // first token whose y this workgroup stores
    const int cb = wg % ncb;
    wg /= ncb;
    const int g = wg % p.groups_b;
    const int b = wg / p.groups_b;
    const int cbase = g * dpg + cb * CPW;    // first channel of this workgroup
    const int nvalid = FAST ? CPW : min(CPW, dpg - cb * CPW);

    const size_t row0 = (static_cast<size_t>(b) * p.dim + cbase) * static_cast<size_t>(L);
    const IT *__restrict__ ub = static_cast<const IT *>(p.u) + row0;
    const IT *__restrict__ db = static_cast<const IT *>(p.delta) + row0;
    IT *__restrict__ ob = static_cast<IT *>(p.out) + row0;
    const IT *__restrict__ Bb =
        BVAR ? static_cast<const IT *>(p.B) + (static_cast<size_t>(b) * p.groups_b + g) * static_cast<size_t>(N) * L
             : nullptr;
    const IT *__restrict__ Cb =
        CVAR ? static_cast<const IT *>(p.C) + (static_cast<size_t>(b) * p.groups_c + (BVAR ? g : 0)) * static_cast<size_t>(N) * L
             : nullptr;
    const float *const Bw = static_cast<const float *>(p.B);   // constant B/C: fp32 weights
    const float *const Cw = static_cast<const float *>(p.C);

    // ---- per-lane recurrence constants ------------------------------------
    // channel of this lane within the workgroup, and which block of SPL states
    // it holds.  With 8 lanes per channel the lanes of channel c of a wave are
    // c, c+8, ..., c+56 (the layout SwapReduce8x4 reduces over).
    // With 4 lanes per channel they are c, c+16, c+32, c+48.
    constexpr bool kSwap = LPC == 8 || LPC == 4;
    constexpr int kCpWave = 64 / LPC;    // channels per wave
    const int lane = tid & 63;
    const int lc = kSwap ? (tid >> 6) * kCpWave + lane % kCpWave : tid / LPC;
    const int lq = kSwap ? lane / kCpWave : tid % LPC;
    const bool lane_ok = lc < nvalid;
    const int dl = cbase + lc;
    float A2[SPL], h[SPL], bco[SPL], cco[SPL];
#pragma unroll
    for (int j = 0; j < SPL; ++j) {
        const int n = lq * SPL + j;
        const bool ok = lane_ok && n < N;
        const size_t idx = static_cast<size_t>(dl) * N + n;
        A2[j] = ok ? p.A[idx] * kLog2eF : 0.0f;   // A_val *= kLog2e (kernel.cuh:170-178)
        bco[j] = (!BVAR && ok) ? Bw[idx] : 0.0f;
        cco[j] = (!CVAR && ok) ? Cw[idx] : 0.0f;
        if (!BVAR && !CVAR) bco[j] = bco[j] * cco[j];  // B*C folded (kernel.cuh:205-210)
        h[j] = 0.0f;
    }

    // Zero the padded state rows once; tiles only overwrite rows < N.
    if (BVAR)
        for (int i = tid; i < (NP - N) * kRow; i += kThreads) sB[N * kRow + i] = 0.0f;
    if (CLOAD)
        for (int i = tid; i < (NP - N) * kRow; i += kThreads) sC[N * kRow + i] = 0.0f;

    // The records in channel c's rows of segment s2: slot s holds segment s's
    // sum of delta' and its N end states, from the first 4-byte boundary on.
    auto record = [&](int c, int s2, int s) __attribute__((always_inline)) {
        const uintptr_t a = reinterpret_cast<uintptr_t>(ob + static_cast<size_t>(c) * L + static_cast<size_t>(s2) * split.len);
        return reinterpret_cast<float *>((a + 3) & ~static_cast<uintptr_t>(3)) + static_cast<size_t>(s) * (N + 1);
    };
    if constexpr (MODE == kSegOut) {
        if (lane_ok)
            for (int s = 0; s < seg; ++s) {
                const float *rec = record(lc, seg, s);
                const float sum = rec[0];
#pragma unroll
                for (int j = 0; j < SPL; ++j) {
                    const int n = lq * SPL + j;
                    const float end = n < N ? rec[1 + n] : 0.0f;
                    // the decay in two halves: it may leave the range of a
                    // float where its product with h does not; a zero state
                    // stays zero under any growth
                    const float half = __builtin_amdgcn_exp2f(0.5f * (sum * A2[j]));
                    h[j] = h[j] == 0.0f ? end : fmaf(half * h[j], half, end);
                }
            }
    }

    float bias[IPT], dsk[IPT], dsum[IPT];
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
        const int it = tid + k * kThreads;
        const int c = it / kQ4;
        const bool ok = it < ITEMS && c < nvalid;
        bias[k] = (ok && p.delta_bias) ? p.delta_bias[cbase + c] : 0.0f;
        dsk[k] = (ok && p.D) ? p.D[cbase + c] : 0.0f;
        dsum[k] = 0.0f;   // kSegState: sum of delta' over this item's tokens
    }

    // ---- tile loads (global -> registers) ----------------------------------
    // FAST: u, delta and y through raw-buffer descriptors over this
    // workgroup's CPW rows (under 2 GiB, checked by the host); a lane's byte
    // offset is fixed, the tile's goes in the scalar operand, so a tile costs
    // no per-lane address arithmetic.
    constexpr int EB = static_cast<int>(sizeof(IT));
    const int rows_bytes = FAST ? CPW * L * EB : 0;
    const SsRsrc ru = SsRowsRsrc(ub, rows_bytes), rdl = SsRowsRsrc(db, rows_bytes), ryo = SsRowsRsrc(ob, rows_bytes);
    int voff[IPT];
#pragma unroll
    for (int k = 0; k < IPT; ++k) {
        const int it = min(tid + k * kThreads, ITEMS - 1);   // spare lanes re-read a valid item
        voff[k] = ((it / kQ4) * L + (it % kQ4) * 4) * EB;
    }
    // Two register sets of a tile's loads, used in turn by consecutive full
    // tiles, so a prefetch lands where it is consumed (no register copies).
    using R4 = Raw4<IT>;
    R4 uA[IPT], dA[IPT], bcA[BCPT], uB[IPT], dB[IPT], bcB[BCPT];
    auto load_full = [&](int t0, R4 (&ureg)[IPT], R4 (&dreg)[IPT], R4 (&bcreg)[BCPT])
                         __attribute__((always_inline)) {   // FAST, whole tile in range: no guards
#pragma unroll
        for (int k = 0; k < IPT; ++k) {
            ureg[k] = SsBufLoad4<IT>(ru, voff[k], t0 * EB);
            dreg[k] = SsBufLoad4<IT>(rdl, voff[k], t0 * EB);
        }
        if constexpr (NBC > 0) {
            const int per = N * kQ4;
#pragma unroll
            for (int k = 0; k < BCPT; ++k) {
                const int it = min(tid + k * kThreads, NBC * per - 1);
                const int r = it % per;
                const IT *row = ((BVAR && (!CLOAD || it < per)) ? Bb : Cb) + static_cast<size_t>(r / kQ4) * L;
                bcreg[k] = LoadRaw4(row, t0 + (r % kQ4) * 4);
            }
        }
    };
    auto load_guarded = [&](int t0, F4 (&ureg)[IPT], F4 (&dreg)[IPT], F4 (&bcreg)[BCPT])
                            __attribute__((always_inline)) {   // any tile: clamped addresses, zero past the ends
#pragma unroll
        for (int k = 0; k < IPT; ++k) {
            const int it = tid + k * kThreads;
            const int c = min(it / kQ4, nvalid - 1), t = t0 + (it % kQ4) * 4;
            const bool ok = it < ITEMS && it / kQ4 < nvalid;
            ureg[k] = LoadRow4Guarded(ub + static_cast<size_t>(c) * L, t, L, ok);
            dreg[k] = LoadRow4Guarded(db + static_cast<size_t>(c) * L, t, L, ok);
        }
        if constexpr (NBC > 0) {
            const int per = N * kQ4;
#pragma unroll
            for (int k = 0; k < BCPT; ++k) {
                const int it = min(tid + k * kThreads, NBC * per - 1);
                const int r = it % per;
                const IT *row = ((BVAR && (!CLOAD || it < per)) ? Bb : Cb) + static_cast<size_t>(r / kQ4) * L;
                bcreg[k] = LoadRow4Guarded(row, t0 + (r % kQ4) * 4, L, true);
            }
        }
    };

    // ---- phase 1: bias, softplus, delta*u into LDS; keep D*u ----------------
    F4 skip[IPT];
    auto phase1 = [&](int t0, bool full, const F4 (&ureg)[IPT], F4 (&dreg)[IPT], const F4 (&bcreg)[BCPT])
                      __attribute__((always_inline)) {
        // delta' = softplus?(delta + bias): one uniform branch per tile
        if (p.delta_softplus) {
#pragma unroll
            for (int k = 0; k < IPT; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) dreg[k].v[e] = Softplus(dreg[k].v[e] + bias[k]);
        } else {
#pragma unroll
            for (int k = 0; k < IPT; ++k)
#pragma unroll
                for (int e = 0; e < 4; ++e) dreg[k].v[e] += bias[k];
        }
#pragma unroll
        for (int k = 0; k < IPT; ++k) {
            const int it = tid + k * kThreads;
            if (ITEMS % kThreads == 0 || it < ITEMS) {
                const int c = it / kQ4, q4 = it % kQ4;
                F4 dlv, duv;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float x = dreg[k].v[e];
                    if (!full && t0 + q4 * 4 + e >= L) x = 0.0f;   // past the end: a = 1, b = 0
                    dlv.v[e] = x;
                    duv.v[e] = x * ureg[k].v[e];
                    skip[k].v[e] = dsk[k] * ureg[k].v[e];
                }
                if constexpr (kState) dsum[k] += (dlv.v[0] + dlv.v[1]) + (dlv.v[2] + dlv.v[3]);
                *reinterpret_cast<float4 *>(&sDl[c * kRow + q4 * 4]) = make_float4(dlv.v[0], dlv.v[1], dlv.v[2], dlv.v[3]);
                *reinterpret_cast<float4 *>(&sDu[c * kRow + q4 * 4]) = make_float4(duv.v[0], duv.v[1], duv.v[2], duv.v[3]);
            }
        }
        if constexpr (NBC > 0) {
            const int per = N * kQ4;
#pragma unroll
            for (int k = 0; k < BCPT; ++k) {
                const int it = tid + k * kThreads;
                if (it < NBC * per) {
                    const bool isB = BVAR && (!CLOAD || it < per);
                    const int r = it % per;
                    float *dst = (isB ? sB : sC) + (r / kQ4) * kRow + (r % kQ4) * 4;
                    *reinterpret_cast<float4 *>(dst) = make_float4(bcreg[k].v[0], bcreg[k].v[1], bcreg[k].v[2], bcreg[k].v[3]);
                }
            }
        }
    };

    // ---- phase 2: the recurrence over one tile ------------------------------
    auto phase2 = [&]() __attribute__((always_inline)) {
        const float *rDl = sDl + lc * kRow;
        const float *rDu = sDu + lc * kRow;
        float *rY = sY + lc * kRow;
#pragma unroll
        for (int q4 = 0; q4 < kQ4; ++q4) {
            const float4 dl4 = *reinterpret_cast<const float4 *>(rDl + q4 * 4);
            const float4 du4 = *reinterpret_cast<const float4 *>(rDu + q4 * 4);
            const float dlv[4] = {dl4.x, dl4.y, dl4.z, dl4.w};
            const float duv[4] = {du4.x, du4.y, du4.z, du4.w};
            float y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < SPL; ++j) {
                float bv[4] = {0.0f, 0.0f, 0.0f, 0.0f}, cv[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (BVAR) {
                    const float4 x = *reinterpret_cast<const float4 *>(sB + (lq * SPL + j) * kRow + q4 * 4);
                    bv[0] = x.x; bv[1] = x.y; bv[2] = x.z; bv[3] = x.w;
                }
                if constexpr (CLOAD) {
                    const float4 x = *reinterpret_cast<const float4 *>(sC + (lq * SPL + j) * kRow + q4 * 4);
                    cv[0] = x.x; cv[1] = x.y; cv[2] = x.z; cv[3] = x.w;
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float a = __builtin_amdgcn_exp2f(dlv[e] * A2[j]);
                    const float bt = BVAR ? bv[e] * duv[e] : duv[e];
                    h[j] = fmaf(a, h[j], bt);                 // (a1*a0, a1*b0 + b1)
                    if constexpr (kState) continue;
                    float cc;
                    if constexpr (CVAR) cc = BVAR ? cv[e] : bco[j] * cv[e];
                    else cc = BVAR ? cco[j] : bco[j];
                    y[e] = fmaf(h[j], cc, y[e]);              // out += h * C
                }
            }
            if constexpr (kState) {
            } else if constexpr (LPC == 8) {
                // lanes c and c + 8 hold the same sum for the same slot: both
                // write it (no exec-mask region inside the token loop)
                rY[q4 * 4 + SwapReducedToken(lane)] = SwapReduce8x4(y);
            } else if constexpr (LPC == 4) {
                rY[q4 * 4 + SwapReducedToken(lane)] = SwapReduce4x4(y);   // every lane: a distinct (channel, token)
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    y[e] = LaneGroupSum<LPC>(y[e]);
                    // keep the whole reduction ahead of the branch below, so every
                    // step folds into one v_add_f32_dpp (no instruction emitted)
                    asm volatile("" : "+v"(y[e]));
                }
                if (lq == 0) *reinterpret_cast<float4 *>(rY + q4 * 4) = make_float4(y[0], y[1], y[2], y[3]);
            }
        }
    };

    // ---- phase 3: add D*u, store y -------------------------------------------
    auto phase3 = [&](int t0, bool full) __attribute__((always_inline)) {
        if constexpr (kState) return;
        if (MODE == kSegOut && t0 < y_from) return;
#pragma unroll
        for (int k = 0; k < IPT; ++k) {
            const int it = tid + k * kThreads;
            const int c = it / kQ4, q4 = it % kQ4;
            if ((ITEMS % kThreads == 0 || it < ITEMS) && (FAST || c < nvalid)) {
                F4 acc = skip[k];
                const float4 x = *reinterpret_cast<const float4 *>(sY + c * kRow + q4 * 4);
                acc.v[0] += x.x; acc.v[1] += x.y; acc.v[2] += x.z; acc.v[3] += x.w;
                if (FAST && full) {
                    SsBufStore4<IT>(ryo, voff[k], t0 * EB, acc);
                } else {
                    IT *row = ob + static_cast<size_t>(c) * L;
                    StoreRow4(row, t0 + q4 * 4, L, FAST, acc);
                }
            }
        }
        // sY is rewritten only after the next phase-1 barrier; sDl/sDu/sB/sC
        // were last read before the previous barrier.
    };

    int nfull = FAST ? (te - tb) / kTile : 0;   // tiles taken on the unguarded path
    // a full tile from one register set, prefetching the next tile into the other
    auto full_tile = [&](int i, const R4 (&u)[IPT], const R4 (&d)[IPT], const R4 (&bc)[BCPT], R4 (&nu)[IPT], R4 (&nd)[IPT],
                         R4 (&nbc)[BCPT]) __attribute__((always_inline)) {
        const int t0 = tb + i * kTile;
        F4 uw[IPT], dw[IPT], bcw[BCPT];
#pragma unroll
        for (int k = 0; k < IPT; ++k) {
            uw[k] = Widen4<IT>(u[k]);
            dw[k] = Widen4<IT>(d[k]);
        }
        if constexpr (NBC > 0) {
#pragma unroll
            for (int k = 0; k < BCPT; ++k) bcw[k] = Widen4<IT>(bc[k]);
        }
        phase1(t0, true, uw, dw, bcw);
        __syncthreads();
        if (i + 1 < nfull) load_full(t0 + kTile, nu, nd, nbc);   // prefetch; the tail tile loads after the loop
        phase2();
        __syncthreads();
        phase3(t0, true);
    };
    if constexpr (MODE == kSegOut) {
        if (nfull > 0) load_full(tb, uA, dA, bcA);   // before the wait for the records
        bool finite = true;
#pragma unroll
        for (int j = 0; j < SPL; ++j) finite = finite && isfinite(h[j]);
        const bool wave_finite = __ballot(!finite) == 0;
        if (lane == 0) sY[tid / 64] = wave_finite ? 0.0f : 1.0f;   // next written behind phase 1's barrier
        __syncthreads();
        bool walk = false;
#pragma unroll
        for (int i = 0; i < kThreads / 64; ++i) walk = walk || sY[i] != 0.0f;
        if (__builtin_amdgcn_readfirstlane(walk)) {
            tb = 0;
            nfull = FAST ? te / kTile : 0;
#pragma unroll
            for (int j = 0; j < SPL; ++j) h[j] = 0.0f;
            if (nfull > 0) load_full(0, uA, dA, bcA);
        }
    }
    if (nfull > 0) {   // the only path into the full-tile loop
        if constexpr (MODE != kSegOut) load_full(tb, uA, dA, bcA);
        // A tile is entered with its loads issued before the previous tile's
        // IPT stores (vmcnt counts both).  Dropped stores (beyond the
        // descriptor) after tile 0's loads give the first entry the same
        // order, so the loop head's wait lets the stores run on; with the loads
        // alone on that path (or the guarded path of nfull = 0 merging into
        // it) it waited for every store to complete.  Interleaved A/B: 8 x
        // 5120 x 2048 0.3407 -> 0.3343 ms, 2 x 4096 x 4096 0.2225 -> 0.2131,
        // 4 x 5120 x 2048 0.2045 -> 0.2016 (an unconditional prefetch on top,
        // the last tile reloaded: 0.3323, 0.2295, 0.2012).
        if constexpr (!kState) {
#pragma unroll
            for (int k = 0; k < IPT; ++k) SsBufStore4<IT>(ryo, kSsDropOffset, 0, F4{});
        }
        for (int i = 0;; i += 2) {
            full_tile(i, uA, dA, bcA, uB, dB, bcB);
            if (i + 1 >= nfull) break;
            full_tile(i + 1, uB, dB, bcB, uA, dA, bcA);
            if (i + 2 >= nfull) break;
        }
    }
    for (int t0 = tb + nfull * kTile; t0 < te; t0 += kTile) {   // ragged tail (FAST) or every tile
        F4 uw[IPT], dw[IPT], bcw[BCPT];
        load_guarded(t0, uw, dw, bcw);
        phase1(t0, false, uw, dw, bcw);
        __syncthreads();
        phase2();
        __syncthreads();
        phase3(t0, false);
    }
    if constexpr (kState) {
        // the channel's sum of delta' over its kQ4 items, through sDl (last
        // read before the loop's closing barrier)
#pragma unroll
        for (int k = 0; k < IPT; ++k) {
            const int it = tid + k * kThreads;
            if (ITEMS % kThreads == 0 || it < ITEMS) sDl[(it / kQ4) * kRow + it % kQ4] = dsum[k];
        }
        __syncthreads();
        if (lane_ok) {
            float sum = 0.0f;
#pragma unroll
            for (int i = 0; i < kQ4; ++i) sum += sDl[lc * kRow + i];
            for (int s2 = seg + 1; s2 < split.count; ++s2) {
                float *rec = record(lc, s2, seg);
                if (lq == 0) rec[0] = sum;
#pragma unroll
                for (int j = 0; j < SPL; ++j) {
                    const int n = lq * SPL + j;
                    if (n < N) rec[1 + n] = h[j];
                }
            }
        }
        return;
    }
    // Scan state after the last token (tokens past the end kept it unchanged).
    if (p.last_state != nullptr && lane_ok && te == L) {
#pragma unroll
        for (int j = 0; j < SPL; ++j) {
            const int n = lq * SPL + j;
            if (n < N) p.last_state[(static_cast<size_t>(b) * p.dim + dl) * N + n] = h[j];
        }
    }
}

// Lanes per channel and states per lane, with what the forms cost with variable
// B and C (one MI355X, fitted to 480 runs of 1 to 330 channel blocks x 256 to
// 8192 tokens, fp32 and 16-bit; the fits are within 3 to 10% for the whole pass
// and the segments, up to 20% to 4 states, and 7 to 15% for the
// sequence-parallel kernel).  [0]: unguarded accesses (FAST), [1]: guarded.
// 2 x 4, 4 x 4 and 16 x 1 run only under the ss_lpc override.
struct Config {
    int lpc, spl;
    float whole_ns[2];   // the whole pass, per token
    float walk_us, start_us, seq_ps;   // sequence-parallel kernel: per walk, per 1000 channels, per channel and token
    float split_ps[2];   // segments that fill the chip, per channel and token
    float chain_ns[2];   // segments that do not, per token of one
};
constexpr Config kConfigs[] = {
    {1, 4, {146.0f, 310.0f}, 0.6f, 0.5f, 2.9f, {6.3f, 10.5f}, {250.0f, 470.0f}},
    {2, 4, {105.0f, 160.0f}, 0.85f, 0.5f, 4.8f, {5.5f, 9.0f}, {180.0f, 260.0f}},
    {4, 2, {57.0f, 88.0f}, 0.85f, 0.5f, 4.8f, {4.6f, 8.2f}, {98.0f, 140.0f}},
    {4, 4, {80.0f, 112.0f}, 1.4f, 0.9f, 8.5f, {8.0f, 11.0f}, {125.0f, 160.0f}},
    {8, 2, {51.0f, 73.0f}, 1.4f, 0.9f, 8.5f, {6.4f, 9.2f}, {80.0f, 103.0f}},
    {16, 1, {45.0f, 64.0f}, 1.4f, 0.9f, 8.5f, {9.0f, 12.0f}, {70.0f, 90.0f}},
    {8, 4, {84.0f, 112.0f}, 1.55f, 1.0f, 15.5f, {11.8f, 12.8f}, {145.0f, 160.0f}},
    {16, 4, {96.0f, 127.0f}, 3.0f, 1.5f, 85.0f, {27.0f, 33.0f}, {160.0f, 203.0f}},
    {16, 8, {262.0f, 347.0f}, 6.0f, 0.0f, 180.0f, {130.0f, 99.0f}, {430.0f, 555.0f}},
    {16, 16, {924.0f, 1085.0f}, 15.0f, 0.0f, 400.0f, {344.0f, 230.0f}, {1400.0f, 1590.0f}},
};
Config Layout(int lpc, int spl) {
    for (const Config &c : kConfigs)
        if (c.lpc == lpc && c.spl == spl) return c;
    return kConfigs[0];
}

// States per lane and lanes per channel by dstate.  The ss_lpc override sets
// the lanes per channel for dstate <= 16 (1, 2, 4, 8 or 16), for tests and tuning.
Config ChooseConfig(int N) {
    if (N <= 16) {
        const int forced = static_cast<int>(GetOverride(kOverrideSsLpc));
        switch (forced) {
            case 4: return N > 8 ? Layout(4, 4) : Layout(4, 2);
            case 8: return Layout(8, 2);
            case 16: return Layout(16, 1);
            case 2: if (N <= 8) return Layout(2, 4); break;
            case 1: if (N <= 4) return Layout(1, 4); break;
            default: break;
        }
        if (N <= 4) return Layout(1, 4);
        // 8 states: 4 x 2 against 2 x 4 (half the waves, each with twice the
        // serial work): 8 x 5120 x 2048 0.311 -> 0.256 ms, 4 x 5120 x 2048
        // 0.214 -> 0.168, 1 x 5120 x 2048 (whole pass) 0.207 -> 0.119
        if (N <= 8) return Layout(4, 2);
        return Layout(8, 2);   // measured: 0.333 ms vs 0.352 ms (4 lanes) at 8 x 5120 x 2048 x 16
    }
    if (N <= 32) return Layout(8, 4);
    if (N <= 64) return Layout(16, 4);
    if (N <= 128) return Layout(16, 8);
    return Layout(16, 16);
}

template <typename IT, int LPC, int SPL, bool BVAR, bool CVAR, bool VEC>
void LaunchOne(const SelectiveScanParams &p, const SegSplit &split, unsigned blocks, hipStream_t stream) {
    if (!(BVAR && CVAR) || split.count <= 1) {   // the split is built for variable B and C
        XM_NOTE_LAUNCH("SelectiveScanFwdKernel", {TypeTag<IT>()}, LPC, SPL, BVAR, CVAR, VEC, kWhole);
        hipLaunchKernelGGL((SelectiveScanFwdKernel<IT, LPC, SPL, BVAR, CVAR, VEC, kWhole>), dim3(blocks), dim3(kThreads), 0,
                           stream, p, split);
        return;
    }
    if constexpr (BVAR && CVAR) {
        XM_NOTE_LAUNCH("SelectiveScanFwdKernel", {TypeTag<IT>()}, LPC, SPL, BVAR, CVAR, VEC, kSegState);
        hipLaunchKernelGGL((SelectiveScanFwdKernel<IT, LPC, SPL, BVAR, CVAR, VEC, kSegState>), dim3(blocks * (split.count - 1)),
                           dim3(kThreads), 0, stream, p, split);
        XM_NOTE_LAUNCH("SelectiveScanFwdKernel", {TypeTag<IT>()}, LPC, SPL, BVAR, CVAR, VEC, kSegOut);
        hipLaunchKernelGGL((SelectiveScanFwdKernel<IT, LPC, SPL, BVAR, CVAR, VEC, kSegOut>), dim3(blocks * split.count),
                           dim3(kThreads), 0, stream, p, split);
    }
}

template <typename IT, int LPC, int SPL, bool VEC>
void LaunchLSV(const SelectiveScanParams &p, const SegSplit &split, unsigned blocks, hipStream_t stream) {
    if (p.b_var && p.c_var) LaunchOne<IT, LPC, SPL, true, true, VEC>(p, split, blocks, stream);
    else if (p.b_var) LaunchOne<IT, LPC, SPL, true, false, VEC>(p, split, blocks, stream);
    else if (p.c_var) LaunchOne<IT, LPC, SPL, false, true, VEC>(p, split, blocks, stream);
    else LaunchOne<IT, LPC, SPL, false, false, VEC>(p, split, blocks, stream);
}

template <typename IT, int LPC, int SPL>
void LaunchLS(const SelectiveScanParams &p, bool vec, const SegSplit &split, unsigned blocks, hipStream_t stream) {
    if (vec) LaunchLSV<IT, LPC, SPL, true>(p, split, blocks, stream);
    else LaunchLSV<IT, LPC, SPL, false>(p, split, blocks, stream);
}

// Every row of the data tensors on a 4-byte boundary: four tokens an access.
bool AllDwordRows(const SelectiveScanParams &p) {
    const size_t row = static_cast<size_t>(p.seqlen) * (p.in_type == XM_ELEM_FLOAT ? 4 : 2);
    return DwordRows(p.u, row) && DwordRows(p.delta, row) && DwordRows(p.out, row) && (!p.b_var || DwordRows(p.B, row)) &&
           (!p.c_var || DwordRows(p.C, row));
}

// The fast path of the layout: its row descriptors span a workgroup's channels' rows, under 2 GiB.
bool FastRows(const SelectiveScanParams &p, int cpw) {
    const long long row = static_cast<long long>(p.seqlen) * (p.in_type == XM_ELEM_FLOAT ? 4 : 2);
    return AllDwordRows(p) && cpw * row < (1LL << 31) && p.dim_per_group % cpw == 0;
}

template <typename IT>
void LaunchTyped(const SelectiveScanParams &p, const Config &cfg, const SegSplit &split, unsigned blocks, hipStream_t stream) {
    const bool vec = FastRows(p, kThreads / cfg.lpc);
    switch (cfg.lpc * 100 + cfg.spl) {
        case 104: LaunchLS<IT, 1, 4>(p, vec, split, blocks, stream); break;
        case 204: LaunchLS<IT, 2, 4>(p, vec, split, blocks, stream); break;
        case 402: LaunchLS<IT, 4, 2>(p, vec, split, blocks, stream); break;
        case 404: LaunchLS<IT, 4, 4>(p, vec, split, blocks, stream); break;
        case 802: LaunchLS<IT, 8, 2>(p, vec, split, blocks, stream); break;
        case 1601: LaunchLS<IT, 16, 1>(p, vec, split, blocks, stream); break;
        case 804: LaunchLS<IT, 8, 4>(p, vec, split, blocks, stream); break;
        case 1604: LaunchLS<IT, 16, 4>(p, vec, split, blocks, stream); break;
        case 1608: LaunchLS<IT, 16, 8>(p, vec, split, blocks, stream); break;
        default: LaunchLS<IT, 16, 16>(p, vec, split, blocks, stream); break;
    }
}

// d_state = 0: no state, y = D * u (zeros without D); reference
// selective_scan_fwd_kernel.cuh:161 (out = D * u) with an empty state loop (:166).
template <typename IT>
__global__ __launch_bounds__(256) void SelectiveScanSkipKernel(SelectiveScanParams p) {
    const size_t total = static_cast<size_t>(p.batch) * p.dim * p.seqlen;
    const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
    const IT *u = static_cast<const IT *>(p.u);
    IT *out = static_cast<IT *>(p.out);
    for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total; i += stride) {
        const int d = static_cast<int>((i / static_cast<size_t>(p.seqlen)) % static_cast<size_t>(p.dim));
        const float dv = p.D != nullptr ? p.D[d] : 0.0f;
        out[i] = FromF<IT>(dv * ToF(u[i]));
    }
}

template <typename IT>
void LaunchSkip(const SelectiveScanParams &p, hipStream_t stream) {
    const size_t total = static_cast<size_t>(p.batch) * p.dim * p.seqlen;
    const size_t blocks = std::min<size_t>((total + 255) / 256, 8192);
    XM_NOTE_LAUNCH("SelectiveScanSkipKernel", {TypeTag<IT>()}, );
    hipLaunchKernelGGL(SelectiveScanSkipKernel<IT>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, p);
}

// True when neither y nor the last state shares memory with an input (B and C
// variable), or with the other: the rows of y can then hold the sequence split's
// records, and the last segment's workgroup may write the last state while other
// segments' still read the channel's inputs (A, of the same size, among them).
bool OutputsApart(const SelectiveScanParams &p) {
    const size_t eb = p.in_type == XM_ELEM_FLOAT ? 4 : 2, f = sizeof(float), dim = static_cast<size_t>(p.dim);
    const size_t rows = p.batch * dim * p.seqlen * eb, bc = static_cast<size_t>(p.batch) * p.dstate * p.seqlen * eb;
    const MemRange y{p.out, rows}, last{p.last_state, p.batch * dim * p.dstate * f};
    return !Overlap(y, last) &&
           !AnyOverlap({y, last}, {{p.u, rows}, {p.delta, rows}, {p.A, dim * p.dstate * f}, {p.B, bc * p.groups_b},
                                   {p.C, bc * p.groups_c}, {p.D, dim * f}, {p.delta_bias, dim * f}});
}

// At most `most` segments whose rows can hold the records; count 1 if none.
SegSplit FitSegments(const SelectiveScanParams &p, long long most, int min_len) {
    const long long eb = p.in_type == XM_ELEM_FLOAT ? 4 : 2;
    for (long long c = std::min<long long>(most, kSplitMax); c >= 2; --c) {
        const int len = static_cast<int>((p.seqlen + c - 1) / c + 31) / 32 * 32;   // a multiple of the tile (16 or 32)
        const int n = (p.seqlen + len - 1) / len;
        const long long last = p.seqlen - static_cast<long long>(n - 1) * len;
        // the records of n - 1 segments, and the step to a 4-byte boundary, in the shortest segment's rows
        if (n >= 2 && len >= min_len && 4 + 4LL * (n - 1) * (p.dstate + 1) <= last * eb) return {n, len};
    }
    return {1, p.seqlen};
}

struct SsPlan {
    bool seq_parallel;   // SelectiveScanSegKernel
    SegSplit split;
};

// The form of a call: the whole pass (one chain of seqlen steps per channel
// block), the sequence-parallel kernel (one workgroup per channel, 1.3 to 1.8
// times the arithmetic), or segments of the whole pass (1.6 times, two
// launches).  With fewer blocks than CUs the whole pass takes its chain's
// time whatever the channels, the other two grow with the channels.  With
// variable B and C the cheapest by the layout's costs runs; with constant ones
// (no segments; the whole pass is 0.2 to 0.9 of its cost, the sequence-parallel
// kernel 0.2 to 0.95) the sequence-parallel kernel wherever there are fewer
// blocks than CUs.  Measured us, whole / sequence-parallel / segments: 1 x 5120
// x 1999 105 / 102 / 78, 1 x 4096 x 1001 56 / 51 / 39, 1 x 1024 x 1999 106 / 27 /
// 35, 1 x 7168 x 512 30 / 42 / 33; bfloat16 rows off 4 bytes, 2 x 4096 x 1999 163 /
// 468 / 126; guarded, 2 x 12745 x 1264 with one state and constant C 423 / 130 / -;
// 64 states, 1 x 2048 x 1999 193 / 486 / 132.  Over 480 such runs the rule's
// choice takes 0.6% more than the best form on average (geometric mean).
// ss_split override: 1 the whole pass, 2 the sequence-parallel kernel, 3
// segments wherever the rows hold their records.
SsPlan ChoosePlan(const SelectiveScanParams &p, const Config &cfg, long long blocks, int64_t forced) {
    const SegSplit whole{1, p.seqlen};
    const bool seg_fits = SelectiveScanSegFits(p), splits = p.b_var && p.c_var && OutputsApart(p);
    if (forced == 1) return {false, whole};
    if (forced == 2) return {seg_fits, whole};
    if (forced == 3) return {false, splits ? FitSegments(p, kSplitMax, 32) : whole};
    if (blocks > kSplitMaxChannelBlocks || p.seqlen < kSegMinSeqlen) return {false, whole};
    const bool seg_ok = seg_fits && blocks < kSegMaxChannelBlocks;
    if (!p.b_var || !p.c_var) return {seg_ok, whole};
    const SegSplit split = splits ? FitSegments(p, kSplitTarget / blocks, kSplitMinLen) : whole;
    const bool f32 = p.in_type == XM_ELEM_FLOAT;
    const int guarded = FastRows(p, kThreads / cfg.lpc) ? 0 : 1;
    const float L = static_cast<float>(p.seqlen);
    const float mch = static_cast<float>(p.batch) * static_cast<float>(p.dim) * 1e-6f;   // million channels: us per ps and token
    // above one block per CU some CUs step two of them
    const float t_whole = 3.0f + 1e-3f * cfg.whole_ns[guarded] * L * (blocks > kSegMaxChannelBlocks ? 1.45f : 1.0f);
    // the sequence-parallel kernel walks blocks of 512 tokens (1024 to 4
    // states, 256 above 16); above 32 states the tokens past the end cost little
    const int walk = p.dstate <= 4 ? 1024 : (p.dstate <= 16 ? 512 : 256);
    const long long walks = (static_cast<long long>(p.seqlen) + walk - 1) / walk;
    const float seq_ps = cfg.seq_ps * (f32 ? 1.0f : (p.dstate <= 32 ? 0.8f : 0.6f));
    // rows off 4 bytes are read token by token, lengths off 4 tokens with a mask
    const float access = !AllDwordRows(p) ? (p.dstate <= 4 ? 2.3f : 3.0f) : (p.seqlen % 4 != 0 ? 1.08f : 1.0f);
    const float t_seq = 2.5f + access * (cfg.walk_us * static_cast<float>(walks) +
                                         mch * (1e3f * cfg.start_us + seq_ps * (p.dstate <= 32 ? static_cast<float>(walks * walk) : L)));
    // the chip's rate or a segment's chain, whichever is longer (a soft maximum), and about 1 us a record to start from
    const float fill = cfg.split_ps[guarded] * (!f32 && p.dstate <= 16 ? 0.9f : 1.0f) * mch * L;
    const float chain = 1e-3f * cfg.chain_ns[guarded] * split.len;
    const float t_split = 4.0f + split.count + std::cbrt(fill * fill * fill + chain * chain * chain);
    if (split.count > 1 && t_split < t_whole && (!seg_ok || t_split < t_seq)) return {false, split};
    return {seg_ok && t_seq < t_whole, whole};
}

}  // namespace

void LaunchSelectiveScan(const SelectiveScanParams &p, void *stream_v) {
    hipStream_t stream = static_cast<hipStream_t>(stream_v);
    if (p.dstate == 0) {
        if (p.in_type == XM_ELEM_FLOAT16) LaunchSkip<_Float16>(p, stream);
        else if (p.in_type == XM_ELEM_BFLOAT16) LaunchSkip<Bf16>(p, stream);
        else LaunchSkip<float>(p, stream);
        XM_LAUNCH_CHECK("SelectiveScanFn (d_state 0)");
        return;
    }
    const Config cfg = ChooseConfig(p.dstate);
    const int cpw = kThreads / cfg.lpc;
    const long long ncb = (p.dim_per_group + cpw - 1) / cpw;
    const long long blocks = ncb * p.groups_b * static_cast<long long>(p.batch);
    const SsPlan plan = ChoosePlan(p, cfg, blocks, GetOverride(kOverrideSsSplit));
    if (plan.seq_parallel) {
        LaunchSelectiveScanSeg(p, stream);
        return;
    }
    const SegSplit &seg = plan.split;
    if (blocks * seg.count > 2147483647LL) throw Error(XM_ERR_INVALID_ARGUMENT, "SelectiveScanFn launch exceeds the grid limit");
    const unsigned nblocks = static_cast<unsigned>(blocks);
    if (p.in_type == XM_ELEM_FLOAT16) LaunchTyped<_Float16>(p, cfg, seg, nblocks, stream);
    else if (p.in_type == XM_ELEM_BFLOAT16) LaunchTyped<Bf16>(p, cfg, seg, nblocks, stream);
    else LaunchTyped<float>(p, cfg, seg, nblocks, stream);
    XM_LAUNCH_CHECK("SelectiveScanFn");
}

}  // namespace xm
