// GatedDeltaNet2Fn forward for a few tokens (decode steps), gfx950.
//
// One launch, no scratch.  With few tokens the call is bound by the state's
// way in and out (2 dk dv floats per (b,h)) and by the launch itself, so the
// state goes straight from HBM into registers, steps through the tokens there
// and goes back: a workgroup owns one (b,h) and 4 CL value columns, thread
// (key group kg, column lane cl) the columns 4 cl .. 4 cl + 3 of the keys kg,
// kg + KG, ...; every load and store is 16 bytes per lane, CL lanes on one
// state row, and all of a thread's loads are in flight at once.  The chunked
// form, by contrast, pads a chunk to 16 tokens, writes its prepared blocks to
// scratch and reads them back in a second launch.
//
// Per token (the evaluation order of gated_deltanet2.hip), with d = exp(g) and
// S the state before the token:
//     e_j = sum_i (beta_i khat_i) (d_i S_ij),  r_j = sum_i qhat_i (d_i S_ij),
//     u_j = w_j v_j - e_j,  o_j = r_j + (qhat . khat) u_j,  S_ij <- d_i S_ij + khat_i u_j.
// The four vectors of up to kTB tokens are prepared in LDS at a time, one wave
// per token, as {d, beta khat, qhat, khat} per key: one 16-byte read serves
// the four columns.  The sums over the keys are a thread's own keys, the lanes
// of a wave on the same columns (lane swaps and row moves), then the waves'
// sums through LDS, every thread adding them in wave order.
//
// Bound by HBM: 32 x 1 token x 16 heads at 128 x 128 moves 69 MB in 11.6 us
// (5.9 TB/s; the chunked form takes 43.1), 32 x 8 heads at 256 x 256 136 MB in
// 22 (73.5), 64 x 16 heads at 320 x 64 174 MB in 27 (100).  1 x 4 heads: 5.4
// us, the launch (22).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "xm_hip.h"
#include "xm_matrix.h"
#include "xm_params.h"

namespace xm {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kTB = 4;               // tokens prepared at a time, one per wave
// Column blocks of 64 from this many on (two per CU), of 32 below: half the
// blocks prepare the same vectors half as often, but with few blocks the
// smaller ones spread over more CUs.  Measured us, 64 / 32 columns: 32 x 4
// tokens x 16 heads at 128 x 128 16.4 / 20.3, 32 x 16 tokens 35 / 47; 2 x 8
// tokens x 8 heads at 256 x 256 13.0 / 10.5, 8 x 1 x 16 heads 6.4 / 5.9.
constexpr long long kStepWideBlocks = 512;
constexpr float kL2Eps = 1.0e-6f;    // reference kL2NormEps (gated_deltanet2_fwd.cu:14)
static_assert(kTB == kWaves, "one wave per token");

// Sum over the lanes CL, 2 CL, ... apart (CL = 8 or 16) of a wave, in every lane.
template <int CL>
__device__ __forceinline__ float KeyGroupSum(float x) {
    if constexpr (CL == 8) x += DppF<0x128>(x);   // row_ror:8
    const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

template <int CL, int KT>   // column lanes of 4 columns, keys per thread
__global__ __launch_bounds__(kThreads) void Gdn2StepKernel(GatedDeltaNet2Params p) {
    constexpr int KG = kThreads / CL;     // key groups
    constexpr int KP = KG * KT;           // padded keys
    constexpr int KL = (KP + 63) / 64;    // keys per lane in the preparation

    __shared__ __attribute__((aligned(16))) float4 sVec[kTB][KP];        // {d, beta khat, qhat, khat}
    __shared__ float sQk[kTB];                                           // qhat . khat
    __shared__ __attribute__((aligned(16))) v4f sPart[2][kWaves][CL][2]; // per wave: e and r of 4 columns

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int cl = tid % CL, kg = tid / CL;
    const int dk = p.dk, dv = p.dv, T = p.seqlen, H = p.nheads;
    const int ncb = (dv + 4 * CL - 1) / (4 * CL);
    // the column blocks of one (b,h) prepare the same vectors: keep them on one XCD
    const int wg = XcdLocalBlock(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
    const int bh = wg / ncb, c0 = (wg % ncb) * 4 * CL + 4 * cl;
    const int b = bh / H, h = bh % H;
    const size_t row0 = static_cast<size_t>(b) * T * H + h;   // token row t: row0 + t H

    // ---- one token's vectors by one wave: loads, then the work on them
    float q[KL], k[KL], g[KL], bt[KL];
    auto load_token = [&](int t) __attribute__((always_inline)) {
        const size_t src = (row0 + static_cast<size_t>(min(t, T - 1)) * H) * dk;
#pragma unroll
        for (int j = 0; j < KL; ++j) {
            const int kd = min(lane + 64 * j, dk - 1);
            q[j] = p.q[src + kd];
            k[j] = p.k[src + kd];
            g[j] = p.g[src + kd];
            bt[j] = p.beta[src + kd];
        }
    };
    auto prepare = [&](int slot) __attribute__((always_inline)) {
        float qs = 0.0f, ks = 0.0f;
#pragma unroll
        for (int j = 0; j < KL; ++j) {
            const bool ok = lane + 64 * j < dk;
            q[j] = ok ? q[j] : 0.0f;
            k[j] = ok ? k[j] : 0.0f;
            qs = fmaf(q[j], q[j], qs);
            ks = fmaf(k[j], k[j], ks);
        }
        float q_mul = p.scale, k_mul = 1.0f;
        if (p.l2norm) {   // reference :58-62
            q_mul *= rsqrtf(WaveSum64(qs) + kL2Eps);
            k_mul = rsqrtf(WaveSum64(ks) + kL2Eps);
        }
        float qk = 0.0f;
#pragma unroll
        for (int j = 0; j < KL; ++j) {
            const int kd = lane + 64 * j;
            const bool ok = kd < dk;
            const float kn = k[j] * k_mul, qn = q[j] * q_mul;
            qk = fmaf(qn, kn, qk);
            // a padded key: no decay of its zero state, no part in the sums
            if (kd < KP) sVec[slot][kd] = make_float4(ok ? expf(g[j]) : 0.0f, ok ? bt[j] * kn : 0.0f, qn, kn);
        }
        qk = WaveSum64(qk);
        if (lane == 0) sQk[slot] = qk;
    };

    // The token loads go out before the state's: they return first, and the
    // vectors are formed while the state is on its way.
    load_token(wave);
    // State rows through a raw-buffer descriptor over the (b,h) state (under 2
    // GiB, checked by the host): rows past dk and columns past dv read zeros.
    // A last group that dv cuts reads the next row's first columns; they stay
    // in their own lanes' columns and are never stored.
    const size_t sbase = static_cast<size_t>(bh) * dk * dv;
    const int sbytes = dk * dv * 4;
    const Rsrc rs = MakeRsrc(p.initial_state != nullptr ? p.initial_state + sbase : p.q, p.initial_state != nullptr ? sbytes : 0);
    auto soff = [&](int j) { return kg + KG * j < dk && c0 < dv ? ((kg + KG * j) * dv + c0) * 4 : kOutOfRange; };
    v4f S[KT];
#pragma unroll
    for (int j = 0; j < KT; ++j) S[j] = BufF4(rs, soff(j), 0);

    // ---- w, v of this thread's columns, and the output row (written by kg 0)
    auto token_cols = [&](const float *x, int t) __attribute__((always_inline)) {
        const Rsrc r = MakeRsrc(x + (row0 + static_cast<size_t>(t) * H) * dv, dv * 4);
        return BufF4(r, c0 * 4, 0);
    };

    for (int t0 = 0; t0 < T; t0 += kTB) {
        if (t0 > 0) {
            __syncthreads();   // the last block's vectors are read
            load_token(t0 + wave);
        }
        if (t0 + wave < T) prepare(wave);
        __syncthreads();
        const int nt = min(kTB, T - t0);
        for (int tt = 0; tt < nt; ++tt) {
            const int t = t0 + tt, buf = t & 1;
            const v4f wv = token_cols(p.w, t) * token_cols(p.v, t);
            v4f e = {0.0f, 0.0f, 0.0f, 0.0f}, r = {0.0f, 0.0f, 0.0f, 0.0f};
            float kh[KT];
#pragma unroll
            for (int j = 0; j < KT; ++j) {
                const float4 x = sVec[tt][kg + KG * j];
                kh[j] = x.w;
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    S[j][c] *= x.x;
                    e[c] = fmaf(x.y, S[j][c], e[c]);
                    r[c] = fmaf(x.z, S[j][c], r[c]);
                }
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                e[c] = KeyGroupSum<CL>(e[c]);
                r[c] = KeyGroupSum<CL>(r[c]);
            }
            if (lane < CL) {
                sPart[buf][wave][cl][0] = e;
                sPart[buf][wave][cl][1] = r;
            }
            __syncthreads();
            e = sPart[buf][0][cl][0];
            r = sPart[buf][0][cl][1];
#pragma unroll
            for (int w = 1; w < kWaves; ++w) {
                e += sPart[buf][w][cl][0];
                r += sPart[buf][w][cl][1];
            }
            const v4f u = wv - e;
#pragma unroll
            for (int j = 0; j < KT; ++j)
#pragma unroll
                for (int c = 0; c < 4; ++c) S[j][c] = fmaf(kh[j], u[c], S[j][c]);
            if (kg == 0) {
                const float qk = sQk[tt];
                float *o = p.out + (row0 + static_cast<size_t>(t) * H) * dv + c0;
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (c0 + c < dv) o[c] = fmaf(qk, u[c], r[c]);
            }
        }
    }

    if (p.final_state != nullptr) {
        float *fs = p.final_state + sbase;
        const Rsrc rf = MakeRsrc(fs, sbytes);
        if (c0 + 4 <= dv) {
#pragma unroll
            for (int j = 0; j < KT; ++j) BufStF4(rf, soff(j), S[j]);   // rows past dk are dropped
        } else {
#pragma unroll
            for (int j = 0; j < KT; ++j)
#pragma unroll
                for (int c = 0; c < 3; ++c)
                    if (c0 + c < dv) BufStF(rf, soff(j) + (kg + KG * j < dk ? 4 * c : 0), S[j][c]);
        }
    }
}

template <int CL, int KT>
void LaunchStep(const GatedDeltaNet2Params &p, hipStream_t stream) {
    const long long blocks = static_cast<long long>(p.batch) * p.nheads * ((p.dv + 4 * CL - 1) / (4 * CL));
    if (blocks > 2147483647LL) throw Error(XM_ERR_INVALID_ARGUMENT, "GatedDeltaNet2Fn launch exceeds the grid limit");
    XM_NOTE_LAUNCH("Gdn2StepKernel", {}, CL, KT);
    hipLaunchKernelGGL((Gdn2StepKernel<CL, KT>), dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, stream, p);
}

template <int CL>
void LaunchStepKeys(const GatedDeltaNet2Params &p, hipStream_t stream) {
    constexpr int KG = kThreads / CL;
    const int kt = (p.dk + KG - 1) / KG;
    if (kt <= 128 / KG) {
        if (kt <= 64 / KG) LaunchStep<CL, 64 / KG>(p, stream);
        else LaunchStep<CL, 128 / KG>(p, stream);
    } else if (kt <= 192 / KG) LaunchStep<CL, 192 / KG>(p, stream);
    else if (kt <= 256 / KG) LaunchStep<CL, 256 / KG>(p, stream);
    else if (kt <= 320 / KG) LaunchStep<CL, 320 / KG>(p, stream);
    else if (kt <= 384 / KG) LaunchStep<CL, 384 / KG>(p, stream);
    else LaunchStep<CL, 512 / KG>(p, stream);
}

long long WideBlocks(const GatedDeltaNet2Params &p) {
    return static_cast<long long>(p.batch) * p.nheads * ((p.dv + 63) / 64);
}

// With the chip full a block's tokens take turns, while the chunked path's time
// hardly depends on how full its chunk is: many small heads are cheaper there
// from some tokens on.  Both in us, fitted to 500 to 3072 heads of 16 to 512 keys
// x 8 to 64 columns (within 15%).  Measured, chunked / here: 3072 heads of 16 x 16,
// 4 tokens 23 / 18, 8 24 / 30, 16 23 / 54; of 128 x 64, 16 tokens 137 / 105; 1024 of
// 512 x 16, 6 tokens 80 / 71, 12 88 / 118.  Above 384 keys the state leaves room
// for two waves per SIMD.
bool StepIsCheaper(const GatedDeltaNet2Params &p) {
    const double dk = p.dk, rows = static_cast<double>(p.batch) * p.nheads * 1e-3;   // thousands
    const double state_us = rows * dk * p.dv * 8e-3 / 3.0;                            // in and out at 3 TB/s
    const double chunked = 16.0 + 0.055 * dk + 0.04 * dk * rows + state_us;
    const double block_us = p.dk > 384 ? 7.8 : 0.5 + 0.0087 * std::max(dk, 58.0);     // per token of 1000 blocks
    return 3.0 + 0.3 * state_us + 1e-3 * static_cast<double>(WideBlocks(p)) * block_us * p.seqlen <= chunked;
}

}  // namespace

bool GatedDeltaNet2StepFits(const GatedDeltaNet2Params &p) {
    if (p.cu_seqlens != nullptr || p.batch < 1 || p.seqlen < 1 || p.seqlen > kGdn2StepTokens || p.nheads < 1 || p.dk < 1 ||
        p.dk > kGdn2ChunkKeyLimit || p.dv < 1 || static_cast<long long>(p.dk) * p.dv * 4 >= (1LL << 31))
        return false;
    // Every column block of a (b,h) reads the tokens' whole q, k, g and beta
    // rows: an output over them may change what another block has yet to read.
    // The chunked path has read them all before it writes anything.  A block
    // reads v and w of its own columns token by token, so the output may be v or
    // w itself, but not a shifted part of them.
    const size_t rows = static_cast<size_t>(p.batch) * p.seqlen * p.nheads * sizeof(float);
    const size_t keys = rows * p.dk, cols = rows * p.dv, state = static_cast<size_t>(p.batch) * p.nheads * p.dk * p.dv * sizeof(float);
    if (AnyOverlap({{p.out, cols}, {p.final_state, state}}, {{p.q, keys}, {p.k, keys}, {p.g, keys}, {p.beta, keys}}))
        return false;
    for (const float *x : {p.v, p.w})
        if (p.out != x && Overlap({p.out, cols}, {x, cols})) return false;
    for (Override o : {kOverrideGdn2Path, kOverrideGdn2Pairwise, kOverrideGdn2Kpw4, kOverrideGdn2Windowed,
                       kOverrideGdn2Split, kOverrideGdn2Ct})
        if (GetOverride(o) != 0) return false;   // a variant of another path is asked for
    return WideBlocks(p) < kStepWideBlocks || StepIsCheaper(p);
}

bool LaunchGatedDeltaNet2Step(const GatedDeltaNet2Params &p, void *stream_v) {
    if (!GatedDeltaNet2StepFits(p)) return false;
    hipStream_t stream = static_cast<hipStream_t>(stream_v);
    if (WideBlocks(p) >= kStepWideBlocks) LaunchStepKeys<16>(p, stream);
    else LaunchStepKeys<8>(p, stream);
    XM_LAUNCH_CHECK("GatedDeltaNet2Fn (step)");
    return true;
}

}  // namespace xm
