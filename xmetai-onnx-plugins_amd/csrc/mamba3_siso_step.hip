// Mamba3SisoFn forward for a few tokens (decode steps), gfx950.
//
// One launch, no scratch.  With few tokens the call is bound by the state's
// way in and out (2 P N floats per (b,h)) and by the launch, so the state goes
// from HBM into registers, steps through the tokens and goes back: a workgroup
// owns one (b,h) and 16 RP state rows, 16 lanes per row, lane kg the keys
// 4 kg + 64 x .. + 3; every state access is 16 bytes a lane, 256 contiguous
// bytes a row, and all of a thread's loads are in flight at once.  The chunked
// kernel, by contrast, pads the tokens to a chunk of 16 and takes the state in
// 4-byte accesses.
//
// The token recurrence is that of mamba3_siso.hip; the rotation, the angle (in
// turns of the wrap period, fp64) and the per-token scalars are formed as in
// mamba3_siso_chunk.hip.  Tokens are prepared kTB at a time, one wave each, into
// LDS; y goes through LDS and out with the SiLU(Z) gate, one value a thread.
//
// 64 x 128 heads, chunked kernel -> this one: 32 x 1 x 32 heads (72 MB) 68.3 ->
// 14.6 us (4.9 TB/s), 64 x 1 x 32 134 -> 24.4 (5.9 TB/s), 1 x 1 x 32 10.0 -> 6.4
// (the launch), 32 x 16 x 32 72 -> 34.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mamba3_math.h"
#include "xm_hip.h"
#include "xm_matrix.h"
#include "xm_params.h"

namespace xm {
namespace {

using namespace m3;

constexpr int kThreads = 256;
constexpr int kTB = 4;                      // tokens prepared at a time, one per wave
static_assert(kTB == kThreads / 64, "one wave per token");
// Rows per workgroup, by the number of 64-row blocks of the call: 64 rows from
// two blocks per CU on (the vectors are prepared once per block), 32 from half
// a block per CU, else 16 (more CUs share the state and a token's rows).
// Measured us, 16 / 32 / 64 rows, 64 x 128 heads: 32 x 1 x 32 19.6 / 15.9 /
// 14.6, 8 x 1 x 32 8.9 / 7.9 / 7.9, 1 x 8 x 8 8.1 / 8.3 / 10.1.
constexpr long long kBlocks64 = 512, kBlocks32 = 128;
// Tokens: up to one chunk of the chunked kernel (kM3StepTokens), half of one
// where the call has less than a 64-row block per CU: there the chunked kernel
// takes about 10 us whatever the tokens, and 16 tokens here 10 to 12; also where
// a block is mostly padding (up to 16 rows, or 32 keys and less than 64 rows),
// and five with few blocks of up to 32 keys.  Measured us, chunked / here: 298
// heads of 32 x 32, 14 tokens 7.8 / 11.0; 264 of 48 x 32, 16 tokens 10.6 / 13.1;
// 720 of 64 x 32, 16 tokens 19.5 / 17.4; 366 of 16 x 64, 10 tokens 8.0 / 9.1; 104 of
// 64 x 16, 8 tokens 6.0 / 8.4, and 5 tokens of 32 of 96 x 32 5.8 / 5.5.
constexpr long long kBlocksAllTokens = 256;
int TokenLimit(const Mamba3SisoParams &p, long long tall) {
    if (tall < kBlocks32 && p.n <= 32) return 5;
    if (tall < kBlocksAllTokens || p.p <= 16 || (p.n <= 32 && p.p < 64)) return kM3StepTokens / 2;
    return kM3StepTokens;
}

template <int KQ, int RP>   // groups of 64 keys, passes of 16 rows
__global__ __launch_bounds__(kThreads) void Mamba3StepKernel(Mamba3SisoParams p) {
    constexpr int NP = 64 * KQ;             // padded headdim_qk
    constexpr int PB = (KQ + 1) / 2;        // rotation pairs per lane
    constexpr int ROWS = 16 * RP;

    __shared__ __attribute__((aligned(16))) float sQ[kTB][NP], sK[kTB][NP];   // rotated q, k
    __shared__ float sV[kTB][ROWS], sY[kTB][ROWS];
    __shared__ float sScal[kTB][3];                                            // decay, k scale, D + qk gamma

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = tid & 15, rg = tid >> 4;
    const int N = p.n, P = p.p, A = p.a, H = p.nheads, T = p.seqlen;
    const int half_n = N / 2;
    const int nrb = (P + ROWS - 1) / ROWS;
    // the row blocks of one (b,h) prepare the same vectors: keep them on one XCD
    const int wg = XcdLocalBlock(static_cast<int>(blockIdx.x), static_cast<int>(gridDim.x));
    const int rb = wg % nrb, bh = wg / nrb;
    const int b = bh / H, h = bh % H;
    const int gq = h / (H / p.nheads_qk);
    const int r0 = rb * ROWS;
    // Every input through a raw-buffer descriptor: tokens past T, pairs past the
    // end and absent tensors (size 0) read zeros with no branch, so all of a
    // block's loads go out at once (a kernel this short is a few dependent
    // memory latencies long).  The scalar offset is that of a block's first token,
    // which is below the size; what a wave or slot adds to it, and all of an
    // offset into a tensor that may be absent, is per lane.
    const size_t tok0 = static_cast<size_t>(b) * T, sb = static_cast<size_t>(bh) * T;
    auto rows_of = [&](const float *x, size_t first, int stride) {   // token rows of `stride` floats from x + first
        return MakeRsrc(x != nullptr ? x + first : p.DT, x != nullptr ? T * stride * 4 : 0);
    };
    const int qs = p.nheads_qk * N, as = H * A, vs = H * P;
    const Rsrc rq = rows_of(p.Q, (tok0 * p.nheads_qk + gq) * N, qs), rk = rows_of(p.K, (tok0 * p.nheads_qk + gq) * N, qs);
    const Rsrc ra = rows_of(p.Angles, (tok0 * H + h) * A, as);
    const Rsrc rv = rows_of(p.V, (tok0 * H + h) * P, vs), rz = rows_of(p.Z, (tok0 * H + h) * P, vs);
    const Rsrc rdt = rows_of(p.DT, sb, 1), rtr = rows_of(p.Trap, sb, 1), rad = rows_of(p.ADT, sb, 1);
    auto state_of = [&](const float *x, int count) {   // `count` floats of this (b,h), or nothing
        return MakeRsrc(x != nullptr ? x + static_cast<size_t>(bh) * count : p.DT, x != nullptr ? count * 4 : 0);
    };

    // ---- preparation: wave w the token t0 + w; every wave carries the angle
    float2 qv[PB], kv[PB], qb[PB], kb[PB];
    float ang[PB][kTB], dts[kTB], dt0, tr, ad, dt1, tr1, vreg, zreg, dval;
    double carry[PB];
    int poff[PB], aoff[PB];   // this lane's pairs and angles within a token row
#pragma unroll
    for (int x = 0; x < PB; ++x) {
        poff[x] = lane + 64 * x < half_n ? (lane + 64 * x) * 8 : kOutOfRange;
        aoff[x] = lane + 64 * x < A ? (lane + 64 * x) * 4 : kOutOfRange;
    }
    const int vtok = tid / ROWS, vrow = r0 + tid % ROWS;
    const bool vlane = tid < kTB * ROWS && vrow < P;
    auto load_block = [&](int t0) __attribute__((always_inline)) {
        const int t = t0 + wave;
#pragma unroll
        for (int x = 0; x < PB; ++x) {
            qv[x] = BufF2(rq, poff[x] + wave * qs * 4, t0 * qs * 4);
            kv[x] = BufF2(rk, poff[x] + wave * qs * 4, t0 * qs * 4);
#pragma unroll
            for (int s = 0; s < kTB; ++s) ang[x][s] = BufF(ra, aoff[x] + s * as * 4, t0 * as * 4);
        }
#pragma unroll
        for (int s = 0; s < kTB; ++s) dts[s] = BufF(rdt, (t0 + s) * 4);
        // the wave's own token's: picked from dts by the wave index, the compiler
        // would keep dts in LDS at an address from the dispatch packet, which
        // every workgroup would read from host memory (8 x 1 x 32 heads at
        // 64 x 128: 8.5 -> 20 us)
        dt0 = BufF(rdt, t * 4);
        tr = BufF(rtr, t * 4);
        ad = BufF(rad, t * 4);
        dt1 = BufF(rdt, (t + 1) * 4);   // zero past the last token: no look-ahead
        tr1 = BufF(rtr, (t + 1) * 4);
        const int o = vlane ? ((t0 + vtok) * vs + vrow) * 4 : kOutOfRange;
        vreg = BufF(rv, o);
        zreg = BufF(rz, o);
    };
    auto prepare = [&](int t0) __attribute__((always_inline)) {
        float qk = 0.0f;
#pragma unroll
        for (int x = 0; x < PB; ++x) {
            const int pr = lane + 64 * x;
            const bool real = pr < half_n;
            double acc = carry[x], th = 0.0;
#pragma unroll
            for (int s = 0; s < kTB; ++s) {
                acc += static_cast<double>(0.5f * TanhF(ang[x][s])) * static_cast<double>(dts[s]);
                if (s == wave) th = __builtin_amdgcn_fract(acc);   // wrap_two_pi (reference :26-28), in turns
            }
            carry[x] = __builtin_amdgcn_fract(acc);
            const float rev = static_cast<float>(th * kRevPerTurn);
            // a pair without an angle keeps theta = 0: sin 0 = 0, cos 0 = 1
            const float sn = __builtin_amdgcn_sinf(rev), c = __builtin_amdgcn_cosf(rev);
            const float2 q = real ? make_float2(qv[x].x + qb[x].x, qv[x].y + qb[x].y) : make_float2(0.0f, 0.0f);
            const float2 k = real ? make_float2(kv[x].x + kb[x].x, kv[x].y + kb[x].y) : make_float2(0.0f, 0.0f);
            qk = fmaf(q.x, k.x, fmaf(q.y, k.y, qk));   // unrotated q.k (reference :89-106)
            if (pr < NP / 2) {
                *reinterpret_cast<float2 *>(&sQ[wave][2 * pr]) = make_float2(q.x * c - q.y * sn, q.x * sn + q.y * c);
                *reinterpret_cast<float2 *>(&sK[wave][2 * pr]) = make_float2(k.x * c - k.y * sn, k.x * sn + k.y * c);
            }
        }
        qk = WaveSum64(qk);
        const float gam = dt0 * FastSigmoid(tr);
        const float look = dt1 * (1.0f - FastSigmoid(tr1));
        if (lane == 0) {
            sScal[wave][0] = __expf(ad);
            sScal[wave][1] = gam + look;
            sScal[wave][2] = fmaf(qk, gam, dval);
        }
        if (tid < kTB * ROWS) sV[vtok][tid % ROWS] = vreg;
    };

    const Rsrc rqb = MakeRsrc(p.Q_bias + static_cast<size_t>(h) * N, N * 4), rkb = MakeRsrc(p.K_bias + static_cast<size_t>(h) * N, N * 4);
    const Rsrc ria = state_of(p.in_angle, A);
    float angle0[PB];
#pragma unroll
    for (int x = 0; x < PB; ++x) {
        qb[x] = BufF2(rqb, poff[x]);
        kb[x] = BufF2(rkb, poff[x]);
        angle0[x] = BufF(ria, aoff[x]);
    }
    dval = BufF(MakeRsrc(p.D != nullptr ? p.D : p.DT, p.D != nullptr ? H * 4 : 0), h * 4);
    const float tr0 = BufF(rtr, 0);   // the first token's, for the pending look-ahead of the input states
    load_block(0);

    // ---- the state, after the token loads (they return first): rows past P
    // and keys past N read zeros through the descriptor of the (b,h) state
    // (under 2 GiB, checked by the host)
    v4f S[RP][KQ];
    const size_t sbase = static_cast<size_t>(bh) * P * N;
    const int sbytes = P * N * 4;
    auto soff = [&](int x, int y) {
        const int row = r0 + 16 * x + rg, key = 64 * y + 4 * kg;
        return row < P && key < N ? (row * N + key) * 4 : kOutOfRange;
    };
    const Rsrc rs = state_of(p.in_ssm, P * N), rik = state_of(p.in_k, N), riv = state_of(p.in_v, P);
    float vl[RP];
    v4f kl[KQ];
#pragma unroll
    for (int x = 0; x < RP; ++x) {
        vl[x] = BufF(riv, (r0 + 16 * x + rg) * 4);
#pragma unroll
        for (int y = 0; y < KQ; ++y) S[x][y] = BufF4(rs, soff(x, y), 0);
    }
#pragma unroll
    for (int y = 0; y < KQ; ++y) kl[y] = BufF4(rik, (64 * y + 4 * kg) * 4, 0);
    const bool pending = p.in_ssm != nullptr;   // a look-ahead term is still to be added

    for (int t0 = 0; t0 < T; t0 += kTB) {
        if (t0 > 0) {
            load_block(t0);
            __syncthreads();   // the last block's vectors and y are read
        } else {
#pragma unroll
            for (int x = 0; x < PB; ++x) carry[x] = static_cast<double>(angle0[x]) * kInvTwoPiF;
        }
        prepare(t0);
        __syncthreads();
        const int nt = min(kTB, T - t0);
        const float zcur = zreg;
        if (t0 == 0) {
            // S = ssm + v (x) k DT_0 (1 - sigmoid(Trap_0)); a group that N cuts
            // holds the next row's first keys: zero them
            const float look0 = pending ? dts[0] * (1.0f - FastSigmoid(tr0)) : 0.0f;
#pragma unroll
            for (int y = 0; y < KQ; ++y)
#pragma unroll
                for (int x = 0; x < RP; ++x)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float s = 64 * y + 4 * kg + e < N ? S[x][y][e] : 0.0f;
                        S[x][y][e] = fmaf(vl[x], kl[y][e] * look0, s);
                    }
        }
        for (int tt = 0; tt < nt; ++tt) {
            const float dec = sScal[tt][0], ks = sScal[tt][1], diag = sScal[tt][2];
            v4f q[KQ], k[KQ];
#pragma unroll
            for (int y = 0; y < KQ; ++y) {
                q[y] = LdsF4(&sQ[tt][64 * y + 4 * kg]);
                k[y] = LdsF4(&sK[tt][64 * y + 4 * kg]);
            }
#pragma unroll
            for (int x = 0; x < RP; ++x) {
                const float v = sV[tt][16 * x + rg], vk = v * ks;
                float acc = 0.0f;
#pragma unroll
                for (int y = 0; y < KQ; ++y)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        S[x][y][e] *= dec;                       // decay before the readout (reference :140-143)
                        acc = fmaf(q[y][e], S[x][y][e], acc);
                        S[x][y][e] = fmaf(vk, k[y][e], S[x][y][e]);
                    }
                acc = fmaf(diag, v, RowSum16(acc));
                if (kg == 0) sY[tt][16 * x + rg] = acc;
            }
        }
        __syncthreads();
        if (vlane && vtok < nt) {
            float y = sY[vtok][tid % ROWS];
            if (p.Z != nullptr) y *= zcur * FastSigmoid(zcur);   // silu gate (reference :155-158)
            p.out[((tok0 + t0 + vtok) * H + h) * P + vrow] = y;
        }
    }

    if (p.f_ssm == nullptr) return;
    const Rsrc rf = MakeRsrc(p.f_ssm + sbase, sbytes);
#pragma unroll
    for (int x = 0; x < RP; ++x)
#pragma unroll
        for (int y = 0; y < KQ; ++y) {
            const int key = 64 * y + 4 * kg;
            if (key + 4 <= N) {
                BufStF4(rf, soff(x, y), S[x][y]);   // rows past P are dropped
            } else if (key < N && r0 + 16 * x + rg < P) {   // N even: two keys left
                BufStF(rf, soff(x, y), S[x][y][0]);
                BufStF(rf, soff(x, y) + 4, S[x][y][1]);
            }
        }
    if (tid < ROWS && r0 + tid < P) p.f_v[static_cast<size_t>(bh) * P + r0 + tid] = sV[(T - 1) % kTB][tid];
    if (rb == 0) {
        if (wave == 0) {
#pragma unroll
            for (int x = 0; x < PB; ++x)
                if (lane + 64 * x < A)
                    p.f_angle[static_cast<size_t>(bh) * A + lane + 64 * x] = static_cast<float>(carry[x] * kTwoPiF);
        }
        for (int i = tid; i < N; i += kThreads) p.f_k[static_cast<size_t>(bh) * N + i] = sK[(T - 1) % kTB][i];
    }
}

template <int KQ, int RP>
void LaunchStep(const Mamba3SisoParams &p, hipStream_t stream) {
    const long long blocks = static_cast<long long>(p.batch) * p.nheads * ((p.p + 16 * RP - 1) / (16 * RP));
    if (blocks > 2147483647LL) throw Error(XM_ERR_INVALID_ARGUMENT, "Mamba3SisoFn launch exceeds the grid limit");
    XM_NOTE_LAUNCH("Mamba3StepKernel", {}, KQ, RP);
    hipLaunchKernelGGL((Mamba3StepKernel<KQ, RP>), dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, stream, p);
}

template <int RP>
void LaunchStepKeys(const Mamba3SisoParams &p, hipStream_t stream) {
    if (p.n <= 64) LaunchStep<1, RP>(p, stream);
    else if (p.n <= 128) LaunchStep<2, RP>(p, stream);
    else if (p.n <= 192) LaunchStep<3, RP>(p, stream);
    else LaunchStep<4, RP>(p, stream);
}

// Where an output shares memory with an input.
struct OutputSharing {
    bool with_head;   // with an input that every row block of a head reads
    bool out_moves;   // the y rows with those, or with another place of V or Z
};
OutputSharing SharesOf(const Mamba3SisoParams &p) {
    const size_t f = sizeof(float), rows = static_cast<size_t>(p.batch) * p.seqlen;
    const size_t bh = static_cast<size_t>(p.batch) * p.nheads * f, th = rows * p.nheads * f, h = static_cast<size_t>(p.nheads) * f;
    const size_t qk = rows * p.nheads_qk * p.n * f;
    const MemRange out{p.out, th * p.p};
    const std::initializer_list<MemRange> head = {
        {p.Q, qk}, {p.K, qk}, {p.Angles, th * p.a}, {p.ADT, th}, {p.DT, th}, {p.Trap, th}, {p.Q_bias, h * p.n},
        {p.K_bias, h * p.n}, {p.D, h}, {p.in_angle, bh * p.a}, {p.in_k, bh * p.n}};
    OutputSharing s{AnyOverlap({out, {p.f_ssm, bh * p.p * p.n}, {p.f_angle, bh * p.a}, {p.f_k, bh * p.n}, {p.f_v, bh * p.p}}, head),
                    AnyOverlap({out}, head)};
    for (const float *x : {p.V, p.Z}) s.out_moves = s.out_moves || (p.out != x && Overlap(out, {x, th * p.p}));
    return s;
}

}  // namespace

bool LaunchMamba3SisoStep(const Mamba3SisoParams &p, void *stream_v) {
    if (p.cu_seqlens != nullptr || p.seqlen < 1 || p.seqlen > kM3StepTokens || p.n > 256 || p.batch < 1 ||
        static_cast<long long>(p.p) * p.n * 4 >= (1LL << 31) ||
        std::max({static_cast<long long>(p.nheads_qk) * p.n, static_cast<long long>(p.nheads) * p.a,
                  static_cast<long long>(p.nheads) * p.p}) * 4 * (p.seqlen + kTB) >= (1LL << 31) ||
        GetOverride(kOverrideM3Path) != 0)
        return false;
    const OutputSharing shares = SharesOf(p);
    // A block takes its tokens kTB at a time: what it writes of the first ones
    // must not be an input of later ones.
    if (shares.out_moves && p.seqlen > kTB) return false;
    // Above 64 rows a head has several row blocks: none may write what another
    // has yet to read (final states over the input states, for instance).
    if (shares.with_head && p.p > 64) return false;
    const int one_block = shares.with_head ? p.p : 0;   // rows that must be one block's
    const long long tall = static_cast<long long>(p.batch) * p.nheads * ((p.p + 63) / 64);
    if (p.seqlen > TokenLimit(p, tall) && one_block <= 32) return false;
    hipStream_t stream = static_cast<hipStream_t>(stream_v);
    if (tall >= kBlocks64 || one_block > 32) LaunchStepKeys<4>(p, stream);
    else if (tall >= kBlocks32 || one_block > 16) LaunchStepKeys<2>(p, stream);
    else LaunchStepKeys<1>(p, stream);
    XM_LAUNCH_CHECK("Mamba3SisoFn (step)");
    return true;
}

}  // namespace xm
