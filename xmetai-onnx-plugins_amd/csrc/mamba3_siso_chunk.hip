// Mamba3SisoFn forward, chunked form on fp32 MFMA (gfx950, wave64).
//
// The recurrence (reference mamba3_siso_fwd.cu:79-171), per (b,h) with state
// S [P,N]: S *= e^{ADT_t}; y_t = q^_t . S + (D + qk_t gamma_t) v_t;
// S += v_t (x) k^_t w_t, with q^/k^ the rotated q/k, qk_t the unrotated dot
// product and w_t = gamma_t + look_t (gamma_t = DT_t sigmoid(Trap_t), look_t =
// DT_{t+1} (1 - sigmoid(Trap_{t+1})), 0 for the last token).  The decay is a
// scalar per token, so over a chunk of kC = 16 tokens with cum_t the
// inclusive sum of ADT from the chunk start the recurrence unrolls into
// matrix products:
//   y_t    = e^{cum_t} q^_t . S_prev + sum_{s<t} e^{cum_t - cum_s} w_s (q^_t . k^_s) v_s
//            + (D + qk_t gamma_t) v_t
//   S_next = e^{cum_15} S_prev + sum_s e^{cum_15 - cum_s} w_s v_s (x) k^_s
// (equal to the token-by-token recurrence in exact arithmetic).
//
// A workgroup of 8 waves (12 up to 128 keys) owns one (b,h) and 32 state
// rows (two 16-row tiles) and walks the chunks in order.  Waves 0-3 (product
// waves) form the matrix products and keep S^T in MFMA accumulator layout:
// product wave w holds the key blocks [KBW w, KBW (w+1)) of 16 keys; product
// waves 0 and 1 also finish the previous chunk, with the decay mask and the
// q.k sum that product waves 2 and 3 form for them (and, from 192 keys, the
// whole G^T).  The other waves (preparation waves) prepare the next chunk.
// Each SIMD runs one product wave and one or two preparation waves, so the
// preparation's VALU work and the products' MFMA work overlap.  Per chunk, with
// v_mfma_f32_16x16x4_f32 (A[m][k] in lane m+16k, B[k][n] in lane n+16k,
// D[m][n] in lane n+16(m/4), register m%4):
//   G^T = K^ Q^T   over the wave's keys    (partial, summed across the waves)
//   Y   = Q^ S^T   over the wave's keys    (partial, summed across the waves)
//   S^T = e^{cum_15} S^T + K^T V'           (V'_s = e^{cum_15 - cum_s} w_s v_s)
// and, after the barrier, product waves 0 and 1 each finish one 16-row tile
// of the output: Y e^{cum_t} + (G o L) V + diag v, with L_ts = e^{cum_t - cum_s} w_s
// for s < t, then the SiLU(Z) gate and the store.  An S^T tile register is
// exactly the B operand of the Y product (keys 4(lane/16) + register), so the
// state never moves.
//
// Preparation of chunk j+1 (rotated q^ and k^, V, per-token scalars) runs
// while chunk j's products are formed: the q^ / k^ tiles into one of two LDS
// buffers (chunk parity; chunk j's are read by its products), V^T and the
// per-token fields into one of three (chunk j-1's are read by the finishing
// waves); one barrier per chunk.  Lane (pair lane pq, token group tg) of preparation wave w rotates the pairs
// w PPW + PL x + pq for tokens TPL tg .. TPL tg + TPL - 1.  The angle of a
// pair is a prefix sum over the chunk (fp64: the token groups' sums are
// scanned across lanes) on top of the carried wrapped angle, wrapped once per
// token with the reference's period 2 (float)pi (equal to its wrap after every
// step in exact arithmetic; mamba3_siso.hip does the same).  It is kept in
// turns of that period, where an increment tanh(a) dt (float)pi is the exact
// double tanh(a) dt / 2 and the wrap is one fract.  Tokens past the end
// of the sequence are identity tokens: zero q, k and v, zero ADT and w.
//
// States, packed sequences and the look-ahead hand-over are those of the
// token-by-token kernel (mamba3_siso.hip), which remains the path under the
// m3_path override.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <type_traits>

#include "mamba3_math.h"
#include "xm_hip.h"
#include "xm_matrix.h"
#include "xm_params.h"

namespace xm {
namespace {

using namespace m3;

constexpr int kC = 16;          // tokens per chunk
constexpr int kRows = 32;       // state rows per workgroup (two 16-row tiles)
constexpr int kStateRows = 64; // state rows per workgroup of the sequence split's state launch
constexpr int kBufs = 3;        // chunk buffers: preparing j+1, products of j, finishing j-1
// Row stride (floats) of the [key][token] k^T and [row][token] V^T tiles.
// LDS bank conflicts of the kernel's access patterns, measured per access on
// gfx950 (SQ_LDS_BANK_CONFLICT of a probe issuing each pattern), pitch 20
// against 24: V^T 4-byte stores, 32 rows x 2 tokens per wave, 6 and 14 (8
// rows x 8 tokens: 0 at 24); 16-byte reads of 16 rows x 4 tokens 4 and 0;
// k^T 8-byte stores, 8 pair rows x 8 token pairs per wave, 4 and 12, 0 with
// the k^T tile's 4-token groups XOR-swizzled by (row >> 2) & 3 (KtCol).
constexpr int kTS = kC + 8;
// Physical column of token t in row r of the k^T tile: its 4-token group
// XOR (r >> 2) & 3, so a group's 4 tokens stay contiguous for 16-byte reads.
__device__ __forceinline__ int KtCol(int r, int t) { return (((t >> 2) ^ ((r >> 2) & 3)) << 2) | (t & 3); }

template <int KBW, int NW, int NPW>   // 16-key blocks per product wave, product waves, preparation waves
struct M3CLayout {
    static constexpr int NT = 64 * (NW + NPW);   // threads
    static constexpr int NP = 16 * NW * KBW;     // padded headdim_qk
    static constexpr int PPW = NP / (2 * NPW);   // pairs per preparation wave
    static constexpr int PL = PPW % 16 == 0 ? 16 : 8;   // pair lanes per token group
    static constexpr int PB = PPW / PL;          // pairs per lane
    static constexpr int TG = 64 / PL;           // token groups (4 rows, or 8 half rows)
    static constexpr int TPL = kC / TG;          // tokens per lane
    static constexpr int VPT = kRows * kC / (64 * NPW);   // V values per preparation thread
    // Row stride of the [token][key] q^ tile, 8 floats of padding (NP + 8 is 8
    // modulo 16): row-strided 16-byte accesses on gfx950 run without bank
    // conflicts when the row pitch in floats is 8 times an odd number
    // (measured: pitch 132 doubles both the preparation's paired 8-byte
    // writes, 15.8 against 7.9 LDS cycles per instruction, and the products'
    // 16-byte reads, 7.9 against 4.0).
    static constexpr int QS = NP + 8;
    // A chunk's tiles (floats), double-buffered by chunk parity: only the
    // chunk's products and the next chunk's preparation touch them, and in
    // loops unrolled by two the parity, so every tile address, is a
    // compile-time offset from one per-lane base.
    static constexpr int oQ = 0;                      // q^   [kC][QS]
    static constexpr int oKT = oQ + kC * QS;          // k^T  [NP][kTS]
    static constexpr int oK = oKT + NP * kTS;         // k^   [kC][QS] (KCOPY)
    // A chunk's V^T and per-token fields, in three buffers (the finishing
    // waves read them one chunk later).
    static constexpr int oVT = 0;                     // V^T  [kRows][kTS]
    static constexpr int oCum = oVT + kRows * kTS;    // cum_t
    static constexpr int oEcum = oCum + kC;           // e^{cum_t}
    static constexpr int oW = oEcum + kC;             // w_t = gamma_t + look_t
    static constexpr int oGam = oW + kC;              // gamma_t
    static constexpr int oCs = oGam + kC;             // e^{cum_15 - cum_t} w_t (the update's V' scale)
    static constexpr int oQK = oCs + kC;              // partial q.k per preparation wave [NPW][kC]
    // formed once per chunk for both finishing waves, by product waves 2 and 3
    // while the chunk's products run: the decay mask L_ts = e^{cum_t - cum_s}
    // w_s in the finishing MFMA's A layout (lane t + 16 g, register k: s = 4 g
    // + k; s >= t selected away at use) and D + qk_t gamma_t with qk_t the sum
    // of the q.k partials
    static constexpr int oLm = oQK + NPW * kC;        // [64 lanes][4]
    static constexpr int oDg = oLm + 256;             // D + qk_t gamma_t [kC]
    static constexpr int kSmall = oDg + kC;
    // partial products per parity: [NW][3 tiles: G^T, Y rows 0-15, Y rows 16-31][64 lanes][4]
    static constexpr int kPart = NW * 3 * 64 * 4;
    // k^ also in [token][key] order where LDS holds it (up to 256 keys): the
    // G^T product's A operands then come as one 16-byte read per key block
    // (the q^ tile's conflict-free pattern) instead of four 4-byte reads of k^T
    // (2 conflict cycles each)
    static constexpr bool KCOPY = sizeof(float) * (2 * (oK + kC * QS) + kBufs * kSmall + 2 * kPart) <= 160 * 1024;
    static constexpr int kBig = oK + (KCOPY ? kC * QS : 0);
    static constexpr int oBig = 0, oSmall = 2 * kBig, oPart = oSmall + kBufs * kSmall;
    static constexpr size_t kBytes = sizeof(float) * (oPart + 2 * kPart);
    static_assert(kBig % 4 == 0 && kSmall % 4 == 0 && QS % 4 == 0 && kTS % 4 == 0, "16-byte aligned tiles");
    // the sequence split's state launch keeps only k^T of the tiles and no
    // partial products, and has more state rows
    static constexpr int kStateBig = NP * kTS;
    static constexpr int oStateVT = kSmall, kStateSmall = kSmall + kStateRows * kTS;   // its V^T, behind the fields
    static constexpr size_t kStateBytes = sizeof(float) * (2 * kStateBig + kBufs * kStateSmall);
    static_assert(kBytes <= 160 * 1024, "LDS budget");
    static_assert(PPW % 8 == 0 && PB * PL == PPW && TPL * TG == kC && VPT * 64 * NPW == kRows * kC, "lane mapping");
    static_assert(VPT * NPW == 8 && kRows == 32 && kC == 16, "V^T: 4 row blocks x 2 token blocks of 8 x 8");
};

// Cross-row moves of one fp64 value per lane with the gfx950 lane-swap
// instructions (rows are 16-lane groups r0..r3):
// permlane16_swap(x, x) -> {[x0, x0, x2, x2], [x1, x1, x3, x3]},
// permlane32_swap(x, x) -> {[x0, x1, x0, x1], [x2, x3, x2, x3]}.
struct D2 {
    double a, b;
};
__device__ __forceinline__ D2 Swap16(double x) {
    const unsigned lo = static_cast<unsigned>(__double_as_longlong(x));
    const unsigned hi = static_cast<unsigned>(static_cast<unsigned long long>(__double_as_longlong(x)) >> 32);
    const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    return {__longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(h[0]) << 32) | l[0])),
            __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(h[1]) << 32) | l[1]))};
}
__device__ __forceinline__ D2 Swap32(double x) {
    const unsigned lo = static_cast<unsigned>(__double_as_longlong(x));
    const unsigned hi = static_cast<unsigned>(static_cast<unsigned long long>(__double_as_longlong(x)) >> 32);
    const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    return {__longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(h[0]) << 32) | l[0])),
            __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(h[1]) << 32) | l[1]))};
}
// Exclusive prefix over the rows: [0, a0, a0 + a1, (a0 + a1) + a2] for row values a_r.
__device__ __forceinline__ double RowExclusiveScan(double a, int row) {
    const D2 p = Swap16(a);                 // [a0, a0, a2, a2], [a1, a1, a3, a3]
    const double pair = p.a + p.b;          // [a0+a1, a0+a1, a2+a3, a2+a3]
    const double e1 = (row & 1) ? p.a : 0.0;
    const double lo = Swap32(pair).a;       // a0 + a1 in every row
    return row >= 2 ? lo + e1 : e1;
}
// Exclusive prefix over 8 token groups laid out as half rows (lane l holds
// group 2 (l / 16) + (l / 8) % 2): the partner half row by DPP row_ror:8,
// then the row sums across rows.
__device__ __forceinline__ double DppRor8(double x) {
    const long long v = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_mov_dpp(static_cast<int>(v), 0x128, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(static_cast<int>(v >> 32), 0x128, 0xf, 0xf, true);
    return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}
__device__ __forceinline__ double HalfRowExclusiveScan(double a, int lane);
// Row 3's value in every row.
__device__ __forceinline__ double RowBroadcast3(double x) {
    return Swap16(Swap32(x).b).b;           // [x2, x3, x2, x3] -> [x3, x3, x3, x3]
}
__device__ __forceinline__ double HalfRowExclusiveScan(double a, int lane) {
    const double partner = DppRor8(a);
    const bool upper = (lane & 8) != 0;
    return RowExclusiveScan(a + partner, lane >> 4) + (upper ? partner : 0.0);
}

// Inclusive prefix sum over the 16 lanes of each row (DPP row shifts; a lane
// whose source is outside the row adds 0).
__device__ __forceinline__ float RowInclusiveScan16(float x) {
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x111, 0xf, 0xf, false));   // row_shr:1
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x112, 0xf, 0xf, false));   // row_shr:2
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x114, 0xf, 0xf, false));   // row_shr:4
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x118, 0xf, 0xf, false));   // row_shr:8
    return x;
}

// ---------------------------------------------------------------------------
// Sequence split, for calls whose (b,h) row blocks are fewer than the CUs: a
// workgroup walks its sequence's chunks in order, so such a call takes one
// walk's time on part of the chip.  The decay is a scalar per token, so a
// segment maps its start state S to D S + E, with D the exponential of its sum
// of ADT and E its end state from zero.  The angles are sums over the tokens and
// a rotation by a sum of angles is the product of the rotations, so E is formed
// with the angles counted from the segment's start and turned by the start
// angles afterwards.  Three launches:
//  1. Mamba3ChunkKernel<kM3State>: E, the angle sums (fp64, in turns) and the
//     sum of ADT of every fine segment that another follows (segment 0 from
//     the true start state and angles); k^ alone is rotated, no q, no output.
//  2. Mamba3SegCombineKernel: start states and start angles of the output
//     segments, in segment order.
//  3. Mamba3ChunkKernel<kM3Out>: every output segment from its start state.
// The records live in the output rows of the segment that starts at the same
// token (columns of the row block: 4 bytes x W), which only launch 3's
// workgroup of that segment and row block overwrites, after it has read them:
// no scratch.  A record is the S^T tiles in lane order, the fine segment's
// angle sums, its sum of ADT, the start angles, and a flag per 64 quads of the
// start state: one of them is not finite.  A turn would mix an infinity of one
// key into the key beside it, so a segment whose start state is not finite walks
// the sequence from its first token instead and stores only its own rows.
// Packed sequences split likewise, each by its own length.
// ---------------------------------------------------------------------------
enum M3Mode { kM3Whole, kM3State, kM3Out };
struct M3Split {
    int ls, lf;    // tokens per output segment and per fine segment (multiples of kC; ls a multiple of lf)
    int need;      // tokens a record takes: the last segment has at least these
    int maxseg;    // output segments of a sequence of seqlen tokens
    // output segments of a sequence of T tokens
    __host__ __device__ int Segments(int T) const { return T < ls + need ? 1 : (T - need) / ls + 1; }
};
// Tokens a record needs with NP padded keys at 16 or 32 columns.
constexpr int M3RecordTokens(int np) { return np + np / 8 + 16; }
// The record of the segment starting at token tok (in [B*T]): float e of the
// columns r0 .. r0 + W - 1 of head h.
struct M3Record {
    float *base;
    size_t row;   // floats per token row
    int w;        // columns, 16 or 32
    int np;       // padded keys
    __device__ __forceinline__ float *At(int e) const { return base + static_cast<size_t>(e / w) * row + e % w; }
    __device__ __forceinline__ float *State(int q) const { return At(4 * q); }              // 4 floats, q < np w / 4
    __device__ __forceinline__ int AngleSum(int a) const { return np * w + 2 * a; }        // two words of a double
    __device__ __forceinline__ int DecaySum() const { return np * w + np; }
    __device__ __forceinline__ int StartAngle(int a) const { return np * w + np + 16 + 2 * a; }
    __device__ __forceinline__ int Flags() const { return np * w / 256; }                   // at most 32
    __device__ __forceinline__ float *Flag(int i) const { return At(np * w + 2 * np + 16 + i); }
    __device__ __forceinline__ double GetD(int e) const {
        const unsigned lo = __float_as_uint(*At(e)), hi = __float_as_uint(*At(e + 1));
        return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
    }
    __device__ __forceinline__ void PutD(int e, double x) const {
        const unsigned long long v = static_cast<unsigned long long>(__double_as_longlong(x));
        *At(e) = __uint_as_float(static_cast<unsigned>(v));
        *At(e + 1) = __uint_as_float(static_cast<unsigned>(v >> 32));
    }
};
typedef float v4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ M3Record RecordAt(const Mamba3SisoParams &p, size_t tok, int h, int r0, int np) {
    return {p.out + (tok * p.nheads + h) * p.p + r0, static_cast<size_t>(p.nheads) * p.p, min(kRows, p.p - r0), np};
}
// A sequence's tokens: first (in [B*T]) and count.
struct M3Range {
    size_t tok0;
    int T;
};
__device__ __forceinline__ M3Range RangeOf(const Mamba3SisoParams &p, int b) {
    if (p.cu_seqlens == nullptr) return {static_cast<size_t>(b) * p.seqlen, p.seqlen};
    const long long lo = min(max(p.cu_seqlens[b], 0LL), static_cast<long long>(p.seqlen));
    const long long hi = min(max(p.cu_seqlens[b + 1], lo), static_cast<long long>(p.seqlen));
    return {static_cast<size_t>(lo), static_cast<int>(hi - lo)};
}

// Output segments of a sequence of T tokens in this call.  Packed offsets that
// do not rise can give two sequences the same output rows, and so the same
// records: such a call is not split.  (Every lane of the wave calls it.)
__device__ __forceinline__ int SegmentsOf(const Mamba3SisoParams &p, const M3Split &split, int T) {
    if (p.cu_seqlens != nullptr) {
        bool rises = true;
        for (int b = threadIdx.x & 63; b < p.batch; b += 64) rises = rises && p.cu_seqlens[b] <= p.cu_seqlens[b + 1];
        if (__ballot(!rises) != 0) return 1;
    }
    return split.Segments(T);
}

// LONG: some tensor's token rows of one sequence span 2 GiB or more, beyond a
// buffer descriptor's 32-bit range; every chunk then reads and writes through
// descriptors that start at its own first token.
// HASZ: a Z input (the SiLU gate); without one the finishing waves issue no Z
// loads and no gate.
// MODE: the whole sequence, or a launch of the sequence split (above).  PACKED:
// cu_seqlens absent (0), given (1), or seen at run time (2).  A kernel of its own
// leaves the unpacked pass free of the offsets' code (4 x 4096 x 32 heads 365 ->
// 360 us), but with a Z the compiler schedules that kernel worse (380 -> 385, 64
// keys 249 -> 252), so there one kernel serves both.
template <int KBW, int NW, int NPW, bool LONG, bool HASZ, int MODE, int PACKED>
__global__ __launch_bounds__(64 * (NW + NPW)) void Mamba3ChunkKernel(Mamba3SisoParams p, M3Split split) {
    constexpr bool kState = MODE == kM3State;
    using L = M3CLayout<KBW, NW, NPW>;
    static_assert(NW == 4, "product waves 0 and 1 finish, 2 and 3 take shared work off them");
    constexpr int NT = L::NT;
    constexpr int PPW = L::PPW, PL = L::PL, PB = L::PB, TPL = L::TPL, QS = L::QS;
    constexpr int ROWS = kState ? kStateRows : kRows, PT = ROWS / 16;   // state rows, row tiles
    constexpr int VPT = ROWS * kC / (64 * NPW);                          // V values per preparation thread
    constexpr int oVT = kState ? L::oStateVT : L::oVT;

    constexpr int oKT = kState ? 0 : L::oKT, kBig = kState ? L::kStateBig : L::kBig, oSmall = 2 * kBig;

    extern __shared__ __attribute__((aligned(16))) float smem[];
    float *part = smem + (kState ? 0 : L::oPart);   // unused by kState

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool product_wave = wave < NW;
    const int w = product_wave ? wave : wave - NW;   // index within the role
    const int i16 = lane & 15, g4 = lane >> 4;
    const int N = p.n, P = p.p, A = p.a, H = p.nheads;
    const int half_n = N / 2;
    const int nrb = (P + ROWS - 1) / ROWS;
    // the nrb workgroups of one (b,h) prepare the same token vectors: keep them on one XCD
    // (packed sequences: a sequence's heads over all XCDs, XcdSpreadUnit)
    const int wg = XcdLocalBlock(blockIdx.x, gridDim.x);
    const int nseg_wg = MODE == kM3Whole ? 1 : (kState ? (split.maxseg - 1) * (split.ls / split.lf) : split.maxseg);
    const bool packed = PACKED == 1 || (PACKED == 2 && p.cu_seqlens != nullptr);
    int rb = wg % nrb;
    int seg = MODE == kM3Whole ? 0 : (wg / nrb) % nseg_wg;   // fine segment (kM3State) or output segment
    int bh = wg / nrb / nseg_wg;
    int b = bh / H, h = bh % H;
    if (packed) {
        const XcdUnit u = XcdSpreadUnit(blockIdx.x, nrb);   // units: sequence, segment, head
        const int run = u.unit / H;
        if (run >= p.batch * nseg_wg) return;
        rb = u.part;
        h = u.unit - run * H;
        b = run / nseg_wg;
        seg = run - b * nseg_wg;
        bh = b * H + h;
    }
    const int gq = h / (H / p.nheads_qk);
    const int r0 = rb * ROWS;
    const float dval = p.D ? p.D[h] : 0.0f;
    // (RangeOf's arithmetic, written out: through the struct the whole pass
    // measured 1 to 2% slower at 64 keys, the same loops scheduled otherwise)
    int T_ = p.seqlen;
    size_t tok0_ = static_cast<size_t>(b) * T_;    // in [B*T] for Q/K/V/Angles/Z
    size_t sbase_ = static_cast<size_t>(bh) * T_;  // in [B*H*T] for ADT/DT/Trap
    if (packed) {
        const long long lo = min(max(p.cu_seqlens[b], 0LL), static_cast<long long>(p.seqlen));
        const long long hi = min(max(p.cu_seqlens[b + 1], lo), static_cast<long long>(p.seqlen));
        tok0_ = static_cast<size_t>(lo);
        sbase_ = static_cast<size_t>(h) * p.seqlen + static_cast<size_t>(lo);
        T_ = static_cast<int>(hi - lo);
    }
    // The offsets come from a vector load: make the sequence's range
    // wave-uniform so the buffer descriptors built from it stay in SGPRs.
    const int T = __builtin_amdgcn_readfirstlane(T_);
    const size_t tok0 = Uniform64(tok0_), sbase = Uniform64(sbase_);
    // this workgroup's tokens [cs, te) of the sequence (cs a multiple of kC;
    // te too, or the sequence's end)
    int cs = 0, te = T;
    bool last_seg = true;
    if constexpr (MODE != kM3Whole) {
        const int nseg = SegmentsOf(p, split, T);
        if constexpr (kState) {
            cs = seg * split.lf;
            te = cs + split.lf;
            if (te > (nseg - 1) * split.ls) return;   // no segment follows (workgroup-uniform)
        } else {
            if (seg >= nseg) return;
            cs = seg * split.ls;
            last_seg = seg == nseg - 1;
            te = last_seg ? T : cs + split.ls;
        }
    }
    auto record_of = [&](int i) { return RecordAt(p, tok0 + cs, h, r0 + kRows * i, L::NP); };   // its i-th 32 rows'
    const M3Record rec = record_of(0);
    const int y_from = cs;      // first token whose y this workgroup stores
    bool at_start = seg == 0;   // the walk starts with the sequence, from the input states
    float flag = 0.0f;          // kM3Out: a lane's part of the record's
    auto see_flags = [&]() __attribute__((always_inline)) {
        if (__ballot(flag != 0.0f) == 0) return;
        at_start = true;
        cs = 0;
    };
    if constexpr (MODE == kM3Out) {
        if (!at_start && lane < rec.Flags()) flag = *rec.Flag(lane);
        if (product_wave) see_flags();   // the others have loads of their own to send first
    }
    const float *dtr = p.DT + sbase;
    const float *trr = p.Trap + sbase;
    const float *adr = p.ADT + sbase;
    const size_t q_stride = static_cast<size_t>(p.nheads_qk) * N;
    const float *qbase = p.Q + (tok0 * p.nheads_qk + gq) * N;
    const float *kbase = p.K + (tok0 * p.nheads_qk + gq) * N;
    const size_t a_stride = static_cast<size_t>(H) * A;
    const float *abase = p.Angles + (tok0 * H + h) * A;
    const size_t v_stride = static_cast<size_t>(H) * P;
    const size_t vbase = (tok0 * H + h) * P;   // also the output / Z base

    // ---- preparation lanes: pairs w PPW + PL x + pq, tokens TPL tg + s.  Inputs
    // are read with raw buffer loads through per-chunk descriptors that end at
    // the sequence's last token, so tokens past the end, padded pairs (keys
    // >= N) and pairs without an angle (>= A) read zeros with no branch:
    // zero angle increments, zero q/k (padded pairs) and zero DT/ADT/V (a
    // zero w and v make a token past the end an identity token).
    const int pq = lane % PL, tg = lane / PL;
    int pr[PB], qoff[PB][TPL], aoff[PB][TPL];
    float2 qbias[PB], kbias[PB];
    double carry_rec[PB];   // kM3Out: from the record
    double carry[PB];   // wrapped angle after the last prepared token, in turns of the wrap period
#pragma unroll
    for (int x = 0; x < PB; ++x) {
        pr[x] = w * PPW + PL * x + pq;
        const bool real = pr[x] < half_n, rot = pr[x] < A;
        const int pc = min(pr[x], half_n - 1);
        const float2 qb = *reinterpret_cast<const float2 *>(p.Q_bias + static_cast<size_t>(h) * N + 2 * pc);
        const float2 kb = *reinterpret_cast<const float2 *>(p.K_bias + static_cast<size_t>(h) * N + 2 * pc);
        qbias[x] = real ? qb : make_float2(0.0f, 0.0f);
        kbias[x] = real ? kb : make_float2(0.0f, 0.0f);
        carry[x] = (p.in_angle != nullptr && rot) ? static_cast<double>(p.in_angle[static_cast<size_t>(bh) * A + pr[x]]) * kInvTwoPiF : 0.0;
        if constexpr (kState) {
            if (!at_start) carry[x] = 0.0;   // counted from the segment's start
        } else if constexpr (MODE == kM3Out) {
            carry_rec[x] = !product_wave && rot && !at_start ? rec.GetD(rec.StartAngle(pr[x])) : carry[x];
        }
#pragma unroll
        for (int s = 0; s < TPL; ++s) {
            qoff[x][s] = real ? ((TPL * tg + s) * static_cast<int>(q_stride) + 2 * pr[x]) * 4 : kOutOfRange;
            aoff[x][s] = rot ? ((TPL * tg + s) * static_cast<int>(a_stride) + pr[x]) * 4 : kOutOfRange;
        }
    }
    // V values: block w + NPW u of 8 rows x 8 tokens (row block % (ROWS / 8),
    // token block / (ROWS / 8)), lane l: row l / 8, token l % 8 of the block
    int vrow[VPT], vtok[VPT], voff[VPT];
#pragma unroll
    for (int u = 0; u < VPT; ++u) {
        const int blk = w + NPW * u;
        vrow[u] = 8 * (blk % (ROWS / 8)) + (lane >> 3);
        vtok[u] = 8 * (blk / (ROWS / 8)) + (lane & 7);
        voff[u] = r0 + vrow[u] < P ? (vtok[u] * static_cast<int>(v_stride) + r0 + vrow[u]) * 4 : kOutOfRange;
    }
    // Without LONG (the host keeps T * stride * 4 < 2^31): one descriptor per
    // tensor for the whole sequence, ending at its last token; the range
    // check covers the per-lane plus the scalar offset, so a token past the
    // end (and kOutOfRange, which stays below 2^32 with any in-range addend)
    // is out of range.  A lane's place within the chunk is the per-lane
    // offset; the chunk's offset is added to it (off), or, for the
    // preparation's loads (SOFF, all but 192 keys), passed as the scalar
    // offset, which saves a vector add per load (4 x 4096 x 32 heads: 128 keys
    // 0.388 -> 0.371 ms, 64 keys 0.250 -> 0.243, 256 keys 0.772 -> 0.768;
    // 192 keys 0.628 -> 0.639, where it stays off; the output stores and Z
    // loads gain nothing measurable from it).  With LONG each chunk's
    // descriptors start at its first token (the sequence's rows can pass
    // 2 GiB).
    auto seq_bytes = [&](size_t stride) { return static_cast<int>(static_cast<size_t>(T) * stride * 4); };
    // (`rows` tokens from c0: DT and Trap reach one token into the next chunk,
    // the look-ahead of the chunk's last token)
    auto chunk_rsrc = [&](const float *base, size_t stride, int c0, int rows = kC) __attribute__((always_inline)) {
        return MakeRsrc(base + static_cast<size_t>(c0) * stride, static_cast<int>(static_cast<size_t>(min(T - c0, rows)) * stride * 4));
    };
    const Rsrc rq = MakeRsrc(qbase, seq_bytes(q_stride));
    const Rsrc rk = MakeRsrc(kbase, seq_bytes(q_stride));
    const Rsrc ra = MakeRsrc(abase, seq_bytes(a_stride));
    const Rsrc rd = MakeRsrc(dtr, T * 4);
    const Rsrc rt = MakeRsrc(trr, T * 4);
    const Rsrc rad = MakeRsrc(adr, T * 4);
    const Rsrc rv = MakeRsrc(p.V + vbase, seq_bytes(v_stride));
    const int qs4 = static_cast<int>(q_stride) * 4, as4 = static_cast<int>(a_stride) * 4, vs4 = static_cast<int>(v_stride) * 4;
    // per-lane offset + chunk offset, added as unsigned (no signed overflow near 2^31)
    auto off = [](int a, int b) { return static_cast<int>(static_cast<unsigned>(a) + static_cast<unsigned>(b)); };
    constexpr bool SOFF = KBW != 3;
    auto ld = [&](Rsrc r, int v, int c) __attribute__((always_inline)) { return SOFF ? BufF(r, v, c) : BufF(r, off(v, c)); };
    auto ld2 = [&](Rsrc r, int v, int c) __attribute__((always_inline)) { return SOFF ? BufF2(r, v, c) : BufF2(r, off(v, c)); };

    // Raw inputs of one chunk, prefetched two chunks ahead into one of two
    // register sets (chunk parity), or, where registers are short (more than
    // 128 keys), one chunk ahead into one set.
    constexpr bool DB = KBW <= 2;
    // The preparation wave that also forms the per-token scalars (gamma, w,
    // the decay scan and its exponentials).  With 8 preparation waves the one
    // on SIMD 2 (waves w of a role sit on SIMD w % 4), the SIMD a per-wave
    // barrier-arrival trace shows with spare issue (4 x 4096 x 32 heads, 128
    // keys: 0.356 -> 0.354 ms against the last wave, on SIMD 3).  With 4 the
    // last: on SIMD 0 instead, where the trace also showed spare issue, it
    // measured slower (64 keys 0.241 -> 0.265 ms, 192 keys 0.623 -> 0.650,
    // 256 keys 0.754 -> 0.764).
    constexpr int kScalarWave = NPW == 8 ? 6 : NPW - 1;
    struct Raw {
        float2 qv[PB][TPL], kv[PB][TPL];
        float ang[PB][TPL], dts[TPL], vreg[VPT];
        float sdt, strap, sadt, sdt1, strap1;   // preparation wave kScalarWave, lane t < kC
    };
    Raw raw0, raw1;
    auto load_prep = [&](int c0, Raw &r) __attribute__((always_inline)) {
        float2 (&qv)[PB][TPL] = r.qv;
        float2 (&kv)[PB][TPL] = r.kv;
        float (&ang)[PB][TPL] = r.ang;
        float (&dts)[TPL] = r.dts;
        float (&vreg)[VPT] = r.vreg;
        const int cq = LONG ? 0 : c0 * qs4, ca = LONG ? 0 : c0 * as4, cv = LONG ? 0 : c0 * vs4, cd = LONG ? 0 : c0 * 4;
        const Rsrc q_ = LONG ? chunk_rsrc(qbase, q_stride, c0) : rq;
        const Rsrc k_ = LONG ? chunk_rsrc(kbase, q_stride, c0) : rk;
        const Rsrc a_ = LONG ? chunk_rsrc(abase, a_stride, c0) : ra;
        const Rsrc d_ = LONG ? chunk_rsrc(dtr, 1, c0, kC + 1) : rd;
        const Rsrc t_ = LONG ? chunk_rsrc(trr, 1, c0, kC + 1) : rt;
        const Rsrc ad_ = LONG ? chunk_rsrc(adr, 1, c0) : rad;
        const Rsrc v_ = LONG ? chunk_rsrc(p.V + vbase, v_stride, c0) : rv;
#pragma unroll
        for (int s = 0; s < TPL; ++s) {
            dts[s] = ld(d_, (TPL * tg + s) * 4, cd);
#pragma unroll
            for (int x = 0; x < PB; ++x) {
                if constexpr (!kState) qv[x][s] = ld2(q_, qoff[x][s], cq);
                kv[x][s] = ld2(k_, qoff[x][s], cq);
                ang[x][s] = ld(a_, aoff[x][s], ca);
            }
        }
#pragma unroll
        for (int u = 0; u < VPT; ++u) vreg[u] = ld(v_, voff[u], cv);
        // every preparation wave loads them (same load count on every path); wave kScalarWave uses them
        r.sdt = ld(d_, i16 * 4, cd);
        r.strap = ld(t_, i16 * 4, cd);
        r.sadt = ld(ad_, i16 * 4, cd);
        r.sdt1 = ld(d_, (i16 + 1) * 4, cd);
        r.strap1 = ld(t_, (i16 + 1) * 4, cd);
    };

    // rotated q^ / k^ into the tiles bg, the unrotated q.k, V^T and the
    // per-token scalars of the chunk into bf
    auto prep = [&](float *bg, float *bf, const Raw &r) __attribute__((always_inline)) {
        const float2 (&qv)[PB][TPL] = r.qv;
        const float2 (&kv)[PB][TPL] = r.kv;
        const float (&ang)[PB][TPL] = r.ang;
        const float (&dts)[TPL] = r.dts;
        const float (&vreg)[VPT] = r.vreg;
        float qk[TPL];
#pragma unroll
        for (int s = 0; s < TPL; ++s) qk[s] = 0.0f;
#pragma unroll
        for (int x = 0; x < PB; ++x) {
            double pre[TPL], acc = 0.0;
            // The angle in turns of the wrap period 2 (float)pi (reference
            // :26-28): the increment tanh(a) dt (float)pi is tanh(a) dt / 2
            // turns, exact in double (a product of two floats).
#pragma unroll
            for (int s = 0; s < TPL; ++s) {
                acc += static_cast<double>(0.5f * TanhF(ang[x][s])) * static_cast<double>(dts[s]);
                pre[s] = acc;
            }
            // exclusive prefix of the token groups' sums (lanes pq + PL tg)
            double excl;
            if constexpr (PL == 16) excl = RowExclusiveScan(acc, tg);   // token groups are rows
            else excl = HalfRowExclusiveScan(acc, lane);                 // token groups are half rows
            const double base = carry[x] + excl;
            double th = 0.0;
            float kc0[TPL], kc1[TPL];
#pragma unroll
            for (int s = 0; s < TPL; ++s) {
                th = base + pre[s];
                th = __builtin_amdgcn_fract(th);   // wrap_two_pi (reference :26-28), in turns: th - floor(th), kept below 1
                // a pair without an angle keeps theta = 0: sin 0 = 0, cos 0 = 1
                const float rev = static_cast<float>(th * kRevPerTurn);
                const float sn = __builtin_amdgcn_sinf(rev), c = __builtin_amdgcn_cosf(rev);
                const float2 q = kState ? make_float2(0.0f, 0.0f) : make_float2(qv[x][s].x + qbias[x].x, qv[x][s].y + qbias[x].y);
                const float2 k = make_float2(kv[x][s].x + kbias[x].x, kv[x][s].y + kbias[x].y);
                if constexpr (!kState) {
                    qk[s] = fmaf(q.x, k.x, fmaf(q.y, k.y, qk[s]));   // unrotated q.k (reference :89-106)
                    *reinterpret_cast<float2 *>(bg + L::oQ + (TPL * tg + s) * QS + 2 * pr[x]) =
                        make_float2(q.x * c - q.y * sn, q.x * sn + q.y * c);
                }
                kc0[s] = k.x * c - k.y * sn;
                kc1[s] = k.x * sn + k.y * c;
                if constexpr (L::KCOPY && !kState)
                    *reinterpret_cast<float2 *>(bg + L::oK + (TPL * tg + s) * QS + 2 * pr[x]) = make_float2(kc0[s], kc1[s]);
            }
            const int r0k = 2 * pr[x], r1k = 2 * pr[x] + 1;   // this lane's tokens stay in one swizzled group
            if constexpr (TPL == 4) {
                StF4(bg + oKT + r0k * kTS + KtCol(r0k, 4 * tg), v4f{kc0[0], kc0[1], kc0[2], kc0[3]});
                StF4(bg + oKT + r1k * kTS + KtCol(r1k, 4 * tg), v4f{kc1[0], kc1[1], kc1[2], kc1[3]});
            } else {
                *reinterpret_cast<float2 *>(bg + oKT + r0k * kTS + KtCol(r0k, TPL * tg)) = make_float2(kc0[0], kc0[1]);
                *reinterpret_cast<float2 *>(bg + oKT + r1k * kTS + KtCol(r1k, TPL * tg)) = make_float2(kc1[0], kc1[1]);
            }
            // the chunk's last token
            if constexpr (PL == 16) {
                carry[x] = RowBroadcast3(th);
            } else {
                // row 3 holds groups 6 (lower half) and 7; the DPP move runs in
                // every lane before the select (a move inside a branch would
                // read inactive lanes)
                const double v = RowBroadcast3(th);
                const double vr = DppRor8(v);
                carry[x] = (lane & 8) ? v : vr;
            }
        }
        // q.k partial over this wave's pairs, per token
#pragma unroll
        for (int s = 0; s < (kState ? 0 : TPL); ++s) {
            float v = qk[s];
            v += DppF<0xB1>(v);    // quad_perm [1,0,3,2]
            v += DppF<0x4E>(v);    // quad_perm [2,3,0,1]
            v += DppF<0x141>(v);   // row_half_mirror: the 8 lanes of a half row
            if constexpr (PL == 16) v += DppF<0x128>(v);   // row_ror:8
            bf[L::oQK + w * kC + TPL * tg + s] = v;   // every lane of the token group holds the sum
        }
#pragma unroll
        for (int u = 0; u < VPT; ++u) bf[oVT + vrow[u] * kTS + vtok[u]] = vreg[u];
        if (w == kScalarWave) {
            const float gam = r.sdt * FastSigmoid(r.strap);
            const float look = r.sdt1 * (1.0f - FastSigmoid(r.strap1));   // zero DT past the end
            const float cum = RowInclusiveScan16(r.sadt);   // over the chunk's 16 tokens (lanes 0-15)
            const float cum15 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cum), kC - 1));
            if (lane < kC) {
                bf[L::oCum + lane] = cum;
                bf[L::oEcum + lane] = __expf(cum);
                bf[L::oW + lane] = gam + look;
                bf[L::oGam + lane] = gam;
                bf[L::oCs + lane] = __expf(cum15 - cum) * (gam + look);
            }
        }
    };

    // ---- state: S^T tile (key block kb, row tile pt), lane i16 + 16 g4,
    // register r = S[row r0 + 16 pt + i16][key 16 (KBW w + kb) + 4 g4 + r]
    v4f S[KBW][PT];
    {
        const float look0 = (p.in_ssm != nullptr && T > 0) ? dtr[0] * (1.0f - FastSigmoid(trr[0])) : 0.0f;
#pragma unroll
        for (int kb = 0; kb < KBW; ++kb)
#pragma unroll
            for (int pt = 0; pt < PT; ++pt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int row = r0 + 16 * pt + i16, key = 16 * (KBW * w + kb) + 4 * g4 + r;
                    float v = 0.0f;
                    if (product_wave && at_start && p.in_ssm != nullptr && row < P && key < N) {
                        const float vl = p.in_v[static_cast<size_t>(bh) * P + row];
                        const float kl = p.in_k[static_cast<size_t>(bh) * N + key];
                        v = fmaf(vl, kl * look0, p.in_ssm[(static_cast<size_t>(bh) * P + row) * N + key]);
                    }
                    S[kb][pt][r] = v;
                }
        if constexpr (MODE == kM3Out) {
            if (product_wave && !at_start) {
#pragma unroll
                for (int kb = 0; kb < KBW; ++kb)
#pragma unroll
                    for (int pt = 0; pt < PT; ++pt)
                        if (16 * pt < rec.w) S[kb][pt] = *reinterpret_cast<const v4u *>(rec.State(((KBW * w + kb) * (rec.w / 16) + pt) * 64 + lane));
            }
        }
    }

    // ---- products of one chunk: partial G^T and Y to LDS, then the state update
    // G^T = K Q^T is summed over all keys: the finishing waves 0 and 1 form it
    // over the first GK0 of their key blocks only, waves 2 and 3 over theirs
    // and the remaining GX of wave w - 2's.  Measured (4 x 4096 x 32 heads,
    // 2 x at 192 and 256 keys): up to 128 keys nothing moves (one block
    // moved: 0.398 -> 0.421 ms, both: 0.431); at 192 and 256 keys all of
    // them move (0.684 -> 0.628, 0.809 -> 0.763 ms; with the A operands as
    // 4-byte k^T reads, before the k^ copy fitted there: 0.711 -> 0.656,
    // 0.822 -> 0.795, one of three or two of four 0.659, 0.806).
    constexpr int GK0 = KBW <= 2 ? KBW : 0, GX = KBW - GK0;
    auto load_qk = [&](const float *bg, int nb0, float (&q)[4], float (&k)[4]) __attribute__((always_inline)) {
        const v4f q4 = LdsF4(bg + L::oQ + i16 * QS + nb0 + 4 * g4);
        v4f k4;
        if constexpr (L::KCOPY) k4 = LdsF4(bg + L::oK + i16 * QS + nb0 + 4 * g4);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int kr = nb0 + 4 * g4 + ks;
            q[ks] = q4[ks];                                       // q^[t = i16][key nb0 + 4 g4 + ks]
            if constexpr (L::KCOPY) k[ks] = k4[ks];               // k^[s = i16][same key]
            else k[ks] = bg[oKT + kr * kTS + KtCol(kr, i16)];
        }
    };
    auto products = [&](const float *bg, const float *bf, float *pp) __attribute__((always_inline)) {
        float qa[KBW][4], ka[KBW][4], kt[KBW][4], qx[GX > 0 ? GX : 1][4], kx[GX > 0 ? GX : 1][4];
#pragma unroll
        for (int kb = 0; kb < KBW; ++kb) {
            const int nb0 = 16 * (KBW * w + kb);
            if constexpr (!kState) load_qk(bg, nb0, qa[kb], ka[kb]);
            const v4f t4 = LdsF4(bg + oKT + (nb0 + i16) * kTS + KtCol(nb0 + i16, 4 * g4));
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) kt[kb][ks] = t4[ks];   // k^[s = 4 g4 + ks][key nb0 + i16]
        }
        if (!kState && w >= 2) {
#pragma unroll
            for (int x = 0; x < GX; ++x) load_qk(bg, 16 * (KBW * (w - 2) + GK0 + x), qx[x], kx[x]);
        }
        const v4f cs = LdsF4(bf + L::oCs + 4 * g4);
        const float ecum15 = bf[L::oEcum + kC - 1];
        v4f vt[PT];
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) vt[pt] = LdsF4(bf + oVT + (16 * pt + i16) * kTS + 4 * g4);

        if constexpr (!kState) {
            v4f gp = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int kb = 0; kb < GK0; ++kb)
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) gp = Mfma(ka[kb][ks], qa[kb][ks], gp);   // G^T[s][t]
            if (w >= 2) {
#pragma unroll
                for (int kb = GK0; kb < KBW; ++kb)
#pragma unroll
                    for (int ks = 0; ks < 4; ++ks) gp = Mfma(ka[kb][ks], qa[kb][ks], gp);
#pragma unroll
                for (int x = 0; x < GX; ++x)
#pragma unroll
                    for (int ks = 0; ks < 4; ++ks) gp = Mfma(kx[x][ks], qx[x][ks], gp);
            }
            v4f yp[2];
#pragma unroll
            for (int pt = 0; pt < 2; ++pt) {
                yp[pt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int kb = 0; kb < KBW; ++kb)
#pragma unroll
                    for (int ks = 0; ks < 4; ++ks) yp[pt] = Mfma(qa[kb][ks], S[kb][pt][ks], yp[pt]);   // Y[t][row]
            }
            if (GK0 > 0 || w >= 2) StF4(pp + ((w * 3 + 0) * 64 + lane) * 4, gp);
            StF4(pp + ((w * 3 + 1) * 64 + lane) * 4, yp[0]);
            StF4(pp + ((w * 3 + 2) * 64 + lane) * 4, yp[1]);
        }

        // S^T = e^{cum_15} S^T + K^T V',  V'[s][row] = e^{cum_15 - cum_s} w_s v_s[row]
#pragma unroll
        for (int pt = 0; pt < PT; ++pt) {
            float vs[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) vs[r] = vt[pt][r] * cs[r];
#pragma unroll
            for (int kb = 0; kb < KBW; ++kb) {
                S[kb][pt] *= ecum15;
#pragma unroll
                for (int ks = 0; ks < 4; ++ks) S[kb][pt] = Mfma(kt[kb][ks], vs[ks], S[kb][pt]);
            }
        }
    };

    // ---- output rows 16 pt .. 16 pt + 15 of the chunk at c0 (product waves 0 and 1)
    const int orow = r0 + 16 * w + i16;
    int ooff[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        ooff[r] = (w < 2 && orow < P) ? ((4 * g4 + r) * static_cast<int>(v_stride) + orow) * 4 : kOutOfRange;
    // Z of the rows a finishing wave stores, loaded before the products so the
    // MFMA work covers the latency.
    const Rsrc rz = MakeRsrc(p.Z != nullptr ? p.Z + vbase : p.out, p.Z != nullptr ? seq_bytes(v_stride) : 0);
    const Rsrc ro = MakeRsrc(p.out + vbase, seq_bytes(v_stride));
    const Rsrc rnone = MakeRsrc(p.out, 0);   // every access dropped
    auto load_z = [&](int c0, float (&zr)[4]) __attribute__((always_inline)) {
        if constexpr (!HASZ) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (LONG) zr[r] = BufF(p.Z != nullptr ? chunk_rsrc(p.Z + vbase, v_stride, c0) : rnone, ooff[r]);
            else zr[r] = BufF(rz, off(ooff[r], c0 * vs4));
        }
    };
    // y of chunk c0 (tokens past the end and rows >= P are dropped).  The
    // values stay in their four registers until every store is issued: a
    // store's data register rewritten behind it waits for the store to
    // complete (stores count in vmcnt on gfx950).
    auto store_y = [&](int c0, const float (&y)[4]) __attribute__((always_inline)) {
        if (MODE == kM3Out && c0 < y_from) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (LONG) BufStF(chunk_rsrc(p.out + vbase, v_stride, c0), ooff[r], y[r]);
            else BufStF(ro, off(ooff[r], c0 * vs4), y[r]);
        }
        asm volatile("" ::"v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]));
    };
    auto finish = [&](const float *bf, const float *pp, const float (&zr)[4], float (&y)[4])
                      __attribute__((always_inline)) {
        const int pt = w;
        constexpr int GW0 = GK0 > 0 ? 0 : 2;   // first wave with a G^T partial
        v4f g = LdsF4(pp + ((GW0 * 3) * 64 + lane) * 4), ys = LdsF4(pp + ((1 + pt) * 64 + lane) * 4);
        const v4f dg4 = LdsF4(bf + L::oDg + 4 * g4);   // D + qk_t gamma_t
        const v4f l4 = LdsF4(bf + L::oLm + lane * 4);
#pragma unroll
        for (int w2 = GW0 + 1; w2 < NW; ++w2) g += LdsF4(pp + ((w2 * 3 + 0) * 64 + lane) * 4);   // product waves' partials
#pragma unroll
        for (int w2 = 1; w2 < NW; ++w2) ys += LdsF4(pp + ((w2 * 3 + 1 + pt) * 64 + lane) * 4);
        const v4f ecum4 = LdsF4(bf + L::oEcum + 4 * g4);
        const v4f vt = LdsF4(bf + L::oVT + (16 * pt + i16) * kTS + 4 * g4);
        // M[t = i16][s = 4 g4 + ks] = G[t][s] e^{cum_t - cum_s} w_s for s < t (A operand)
        float m[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int s = 4 * g4 + ks;
            m[ks] = s < i16 ? g[ks] * l4[ks] : 0.0f;
        }
        // acc[r] (t = 4 g4 + r, this lane's row): e^{cum_t} Y + (D + qk_t gamma_t) v_t
        v4f acc;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = fmaf(ecum4[r], ys[r], dg4[r] * vt[r]);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) acc = Mfma(m[ks], vt[ks], acc);   // + sum_{s<t} M[t][s] v_s
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            y[r] = acc[r];
            if constexpr (HASZ) y[r] *= zr[r] * FastSigmoid(zr[r]);   // silu gate (reference :155-158)
        }
    };

    // What both finishing waves of chunk bf would otherwise each form (the
    // finishing waves' SIMDs carry the most issue): wave 2 sums the q.k
    // partials (in preparation-wave order) into D + qk_t gamma_t, wave 3 forms
    // the decay mask, while the chunk's products run; the chunk is finished
    // after the next barrier.
    auto shared_finish = [&](float *bf) __attribute__((always_inline)) {
        if (w == 2) {
            if (lane < kC) {
                float v = bf[L::oQK + lane];
#pragma unroll
                for (int w2 = 1; w2 < NPW; ++w2) v += bf[L::oQK + w2 * kC + lane];
                bf[L::oDg + lane] = fmaf(v, bf[L::oGam + lane], dval);
            }
        } else if (w == 3) {
            const v4f cum4 = LdsF4(bf + L::oCum + 4 * g4), w4 = LdsF4(bf + L::oW + 4 * g4);
            const float cumt = bf[L::oCum + i16];
            v4f l4;
#pragma unroll
            for (int ks = 0; ks < 4; ++ks) l4[ks] = __expf(cumt - cum4[ks]) * w4[ks];
            StF4(bf + L::oLm + lane * 4, l4);
        }
    };

    int nch = (te - cs + kC - 1) / kC;
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    auto big = [&](auto P) { return smem + L::oBig + decltype(P)::value * kBig; };      // chunk parity P
    auto par = [&](auto P) { return part + decltype(P)::value * L::kPart; };
    auto small = [&](int j) { return smem + oSmall + (j % kBufs) * (kState ? L::kStateSmall : L::kSmall); };
    // Each role runs its own loop (the same barriers, in the same order), so
    // the registers one role carries across chunks (the state S; the
    // prefetched inputs and angle carries) never have to coexist, and no wave
    // carries another role's predicated-off work (waves 2 and 3 issue no Z
    // loads or output stores: 0.395 -> 0.387 ms at 4 x 4096 x 32 heads, 128
    // keys).  Iteration j: products of chunk j, finishing of chunk j-1 (waves
    // 0 and 1) or the shared finishing work of chunk j (waves 2 and 3) |
    // prefetch of chunk j+2, preparation of chunk j+1.  Chunk 0's products and
    // the last chunk's finishing are peeled.
    auto prepare_chunks = [&]() __attribute__((always_inline)) {   // the preparation waves' loop
        load_prep(cs, raw0);
        if constexpr (DB) load_prep(cs + min(1, nch - 1) * kC, raw1);
        if constexpr (MODE == kM3Out) {
            see_flags();
            if (cs != y_from) {
                nch = (te + kC - 1) / kC;
                load_prep(0, raw0);
                if constexpr (DB) load_prep(min(1, nch - 1) * kC, raw1);
            } else {
#pragma unroll
                for (int x = 0; x < PB; ++x) carry[x] = carry_rec[x];
            }
        }
        prep(big(P0{}), small(0), raw0);
        if constexpr (!DB) load_prep(cs + min(1, nch - 1) * kC, raw0);
        __syncthreads();
        // unrolled by two for the register sets and the parity (P: chunk j + 1's)
        auto iter = [&](int j, auto P, Raw &ld, const Raw &pr_) __attribute__((always_inline)) {
            if constexpr (DB) load_prep(cs + min(j + 2, nch - 1) * kC, ld);
            prep(big(P), small(j + 1), pr_);
            if constexpr (!DB) load_prep(cs + min(j + 2, nch - 1) * kC, ld);
            __syncthreads();
        };
        if (nch > 1) {
            for (int j = 0;; j += 2) {
                iter(j, P1{}, raw0, DB ? raw1 : raw0);
                if (j + 2 >= nch) break;
                iter(j + 1, P0{}, DB ? raw1 : raw0, raw0);
                if (j + 3 >= nch) break;
            }
        }
        __syncthreads();   // the products of the last chunk
    };
    if constexpr (kState) {
        // the same pipeline without products of q and without finishing: the
        // product waves update the state, the preparation waves run ahead
        if (product_wave) {
            float csum = 0.0f;   // the segment's sum of ADT
            __syncthreads();
            auto step = [&](int j, auto P) __attribute__((always_inline)) {
                csum += small(j)[L::oCum + kC - 1];
                products(big(P), small(j), par(P));
                __syncthreads();
            };
            for (int j = 0; j < nch; j += 2) {
                step(j, P0{});
                if (j + 1 >= nch) break;
                step(j + 1, P1{});
            }
#pragma unroll
            for (int kb = 0; kb < KBW; ++kb)
#pragma unroll
                for (int pt = 0; pt < PT; ++pt) {   // two row tiles to each row block's record
                    if (r0 + 16 * pt >= P) continue;
                    const M3Record rp = record_of(pt / 2);
                    *reinterpret_cast<v4u *>(rp.State(((KBW * w + kb) * (rp.w / 16) + pt % 2) * 64 + lane)) = S[kb][pt];
                }
            if (tid < PT / 2 && r0 + kRows * tid < P) {
                const M3Record rp = record_of(tid);
                *rp.At(rp.DecaySum()) = csum;
            }
            return;
        }
        prepare_chunks();
    } else if (nch > 0 && product_wave && w < 2) {   // workgroup-uniform: an empty sequence passes its states through
        __syncthreads();
        // Z of chunk j is loaded in iteration j (before its products) into
        // the register set of j's parity and gated in iteration j + 1, where
        // chunk j is finished.  Loaded in the finishing iteration itself, it
        // came after the previous chunk's output stores, and the wait for it
        // (stores count in vmcnt on gfx950) waited for those stores to
        // complete.  The sets are written only by the Z loads: a zeroing in
        // every iteration landed on registers the previous stores read.
        float za[4] = {0.0f, 0.0f, 0.0f, 0.0f}, zb[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        load_z(cs, za);
        products(big(P0{}), small(0), par(P0{}));
        __syncthreads();
        // zl: the set for chunk j's Z; zu: chunk j - 1's, finished here.  The
        // values stay in their four registers until every store is issued: a
        // store's data register rewritten behind it waits for the store to
        // complete (stores count in vmcnt on gfx950).
        // P: chunk j's parity.
        auto iter = [&](int j, auto P, float (&zl)[4], const float (&zu)[4]) __attribute__((always_inline)) {
            using Q = std::integral_constant<int, 1 - decltype(P)::value>;
            load_z(cs + j * kC, zl);
            products(big(P), small(j), par(P));
            float y[4];
            finish(small(j - 1), par(Q{}), zu, y);
            store_y(cs + (j - 1) * kC, y);
            __syncthreads();
        };
        for (int j = 1; j < nch; j += 2) {   // unrolled by two for the sets and the parity
            iter(j, P1{}, zb, za);
            if (j + 1 >= nch) break;
            iter(j + 1, P0{}, za, zb);
        }
        float y[4];
        if ((nch - 1) & 1) finish(small(nch - 1), par(P1{}), zb, y);
        else finish(small(nch - 1), par(P0{}), za, y);
        store_y(cs + (nch - 1) * kC, y);
    } else if (nch > 0 && product_wave) {   // waves 2 and 3: products and the shared finishing work
        __syncthreads();
        auto step = [&](int j, auto P) __attribute__((always_inline)) {
            products(big(P), small(j), par(P));
            shared_finish(small(j));
            __syncthreads();
        };
        for (int j = 0; j < nch; j += 2) {   // unrolled by two for the parity
            step(j, P0{});
            if (j + 1 >= nch) break;
            step(j + 1, P1{});
        }
    } else if (nch > 0) {
        prepare_chunks();
    }

    if constexpr (kState) {   // preparation waves: the angles after the segment's last token
#pragma unroll
        for (int x = 0; x < PB; ++x)
            if (tg == 0 && pr[x] < A) {
#pragma unroll
                for (int i = 0; i < ROWS / kRows; ++i)
                    if (r0 + kRows * i < P) record_of(i).PutD(record_of(i).AngleSum(pr[x]), carry[x]);
            }
        return;
    }
    if (p.f_ssm != nullptr && last_seg) {
        if (product_wave) {
#pragma unroll
            for (int kb = 0; kb < KBW; ++kb)
#pragma unroll
                for (int pt = 0; pt < 2; ++pt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = r0 + 16 * pt + i16, key = 16 * (KBW * w + kb) + 4 * g4 + r;
                        if (row < P && key < N) p.f_ssm[(static_cast<size_t>(bh) * P + row) * N + key] = S[kb][pt][r];
                    }
        } else if (rb == 0) {
#pragma unroll
            for (int x = 0; x < PB; ++x)
                if (tg == 0 && pr[x] < A)
                    p.f_angle[static_cast<size_t>(bh) * A + pr[x]] = static_cast<float>(carry[x] * kTwoPiF);
        }
        if (tid < kRows && r0 + tid < P) {
            const size_t o = static_cast<size_t>(bh) * P + r0 + tid;
            p.f_v[o] = T > 0 ? p.V[vbase + static_cast<size_t>(T - 1) * v_stride + r0 + tid]
                             : (p.in_v != nullptr ? p.in_v[o] : 0.0f);
        }
        if (rb == 0) {
            // the last chunk's tiles are intact: its k^T column of the last token
            const int tl = T > 0 ? (T - 1) - cs - (nch - 1) * kC : 0;
            const float *kt = smem + L::oBig + ((nch > 0 ? nch - 1 : 0) & 1) * kBig + oKT;
            for (int i = tid; i < N; i += NT) {
                const size_t o = static_cast<size_t>(bh) * N + i;
                p.f_k[o] = T > 0 ? kt[i * kTS + KtCol(i, tl)] : (p.in_k != nullptr ? p.in_k[o] : 0.0f);
            }
        }
    }
}

// True when no output shares memory with an input, and y none with a final
// state: the rows of y can then hold the sequence split's records, and the last
// segment's workgroup may write the final states while the first segments' read
// the inputs and the input states (a caller may keep both in one buffer).
bool OutputsApart(const Mamba3SisoParams &p) {
    const size_t f = sizeof(float), rows = static_cast<size_t>(p.cu_seqlens != nullptr ? 1 : p.batch) * p.seqlen;
    const size_t bh = static_cast<size_t>(p.batch) * p.nheads * f, th = rows * p.nheads * f, h = static_cast<size_t>(p.nheads) * f;
    const size_t qk = rows * p.nheads_qk * p.n * f;
    const MemRange y{p.out, th * p.p}, ssm{p.f_ssm, bh * p.p * p.n}, angle{p.f_angle, bh * p.a}, k{p.f_k, bh * p.n},
        v{p.f_v, bh * p.p};
    return !AnyOverlap({y}, {ssm, angle, k, v}) &&
           !AnyOverlap({y, ssm, angle, k, v},
                       {{p.Q, qk}, {p.K, qk}, {p.V, th * p.p}, {p.Z, th * p.p}, {p.Angles, th * p.a}, {p.ADT, th}, {p.DT, th},
                        {p.Trap, th}, {p.Q_bias, h * p.n}, {p.K_bias, h * p.n}, {p.D, h},
                        {p.cu_seqlens, (static_cast<size_t>(p.batch) + 1) * sizeof(int64_t)}, {p.in_ssm, bh * p.p * p.n},
                        {p.in_angle, bh * p.a}, {p.in_k, bh * p.n}, {p.in_v, bh * p.p}});
}

// Split when the row blocks fill at most half the CUs, into as many output
// segments as fill them (one workgroup per CU: its registers and LDS admit no
// second), each of as many fine segments as let the state launch fill them too.
// Measured, 64 x 128 heads (us, whole -> split): 1 x 3001 x 32 heads 285 -> 119
// (4 output segments of 2 fine ones; of 1: 143, of 3: 134), 2 x 4096 x 32 388 ->
// 254 (2 of 4; 4 of 1: 295), 1 x 4096 x 8 385 -> 67 (16 of 2), 1 x 1024 x 32 101 ->
// 63, 1 x 600 x 32 63 -> 58; 128 x 256 heads, 1 x 4096 x 16 728 -> 280.  Packed
// sequences, whose lengths the host does not know, split where the whole pass
// fills at most a quarter of the CUs and sequences of even length would gain:
// 4096 tokens in 2 sequences x 8 heads 299 -> 103, 3 x 8 289 -> 147, 2 x 16 301 ->
// 167; above that segments sized by the row can lose (5 x 16 heads of 64 keys 179 ->
// 188).
constexpr long long kSplitBlocks = 256;   // CUs
constexpr int kSplitMax = 16, kFineMax = 8;
M3Split ChooseSplit(const Mamba3SisoParams &p, int np) {
    const M3Split whole{0, 0, 0, 1};
    const int forced = static_cast<int>(GetOverride(kOverrideM3Split));
    if (forced == 1 || p.p % 16 != 0 || !OutputsApart(p)) return whole;
    // a 32-row workgroup of the output launch and a 64-row one of the state
    // launch per CU: one round of each (packed: of the whole row's segments)
    const bool packed = p.cu_seqlens != nullptr;
    const long long bh = static_cast<long long>(packed ? 1 : p.batch) * p.nheads;
    const long long w32 = bh * ((p.p + kRows - 1) / kRows), w64 = bh * ((p.p + kStateRows - 1) / kStateRows);
    const long long walks = packed ? w32 * p.batch : w32;   // workgroups of the whole pass
    if (forced != 2 && walks > (packed ? kSplitBlocks / 4 : kSplitBlocks / 2)) return whole;
    const long long most = std::max<long long>(2, std::min<long long>(kSplitMax, kSplitBlocks / w32));
    const float t_whole = static_cast<float>(p.seqlen) / (packed ? std::max(p.batch, 1) : 1) / kC;
    const int need = M3RecordTokens(np);
    auto up = [](long long x) { return static_cast<int>((x + kC - 1) / kC * kC); };
    for (int s = static_cast<int>(most); s >= 2; --s) {
        const int ls = up((static_cast<long long>(p.seqlen) + s - 1) / s);
        for (int m = static_cast<int>(std::max<long long>(1, std::min<long long>(kFineMax, kSplitBlocks / (w64 * (s - 1))))); m >= 1; --m) {
            const int lf = up((ls + m - 1) / m);
            if (lf < up(need)) continue;
            M3Split split{lf * m, lf, need, 0};
            split.maxseg = split.Segments(p.seqlen);
            if (split.maxseg < 2) continue;
            // in chunk steps: the longest output segment, the fine segment (0.75
            // of a step each) and 12 us of launches (8 steps) against the sequence
            const int out = packed ? split.ls + need : std::max(split.ls, p.seqlen - (split.maxseg - 1) * split.ls);
            const float t_split = (out + 0.75f * lf) / kC + 8.0f;
            if (forced == 2 || t_split < 0.9f * t_whole) return split;
        }
    }
    return whole;
}

// Launch 2 of the sequence split: the start states and start angles of the
// output segments.  A thread takes four state values, two key pairs of one
// row; the end states are read before the start states take their places.
__global__ __launch_bounds__(256) void Mamba3SegCombineKernel(Mamba3SisoParams p, M3Split split, int np, int blocks) {
    const int H = p.nheads, A = p.a;
    const int nrb = (p.p + kRows - 1) / kRows;
    const int blk = blockIdx.x % blocks, rb = blockIdx.x / blocks % nrb, bh = blockIdx.x / blocks / nrb;
    const int b = bh / H, h = bh % H;
    const M3Range r = RangeOf(p, b);
    const int m = split.ls / split.lf, nf = (SegmentsOf(p, split, r.T) - 1) * m;   // fine segments that another follows
    const int q = blk * 256 + threadIdx.x;
    auto record = [&](int f) { return RecordAt(p, r.tok0 + static_cast<size_t>(f) * split.lf, h, rb * kRows, np); };
    const M3Record r0 = record(0);
    if (nf < 1 || q >= np * r0.w / 4) return;
    // tile order: key block, row tile, lane; keys 16 block + 4 (lane / 16) .. + 3
    const int tiles = r0.w / 16, lane = q % 64, key = 16 * (q / 64 / tiles) + 4 * (lane / 16);
    const bool writes_angles = q / 64 % tiles == 0 && lane % 16 == 0;   // one row's threads write their pairs'
    double th[2] = {0.0, 0.0};
    v4f S = {0.0f, 0.0f, 0.0f, 0.0f};   // the state before fine segment f
    // segment f's end state, angle sums and decay, read one segment ahead
    struct Rec {
        v4f end;
        double dth[2];
        float decay;
    };
    auto load = [&](int f) {
        Rec x{{0.0f, 0.0f, 0.0f, 0.0f}, {0.0, 0.0}, 0.0f};
        if (f >= nf) return x;
        const M3Record rf = record(f);
        x.end = *reinterpret_cast<const v4u *>(rf.State(q));
        x.decay = *rf.At(rf.DecaySum());
#pragma unroll
        for (int e = 0; e < 2; ++e)
            if (key / 2 + e < A) x.dth[e] = rf.GetD(rf.AngleSum(key / 2 + e));
        return x;
    };
    Rec next = load(0);
    for (int f = 0; f <= nf; ++f) {
        Rec cur = next;
        next = load(f + 1);
        if (f > 0 && f % m == 0) {
            const M3Record rf = record(f);
            *reinterpret_cast<v4u *>(rf.State(q)) = S;
            const bool inf = !(isfinite(S[0]) && isfinite(S[1]) && isfinite(S[2]) && isfinite(S[3]));
            const bool any = __ballot(inf) != 0;   // whole waves: np w / 4 is a multiple of 64
            if (lane == 0) *rf.Flag(q / 64) = any ? 1.0f : 0.0f;
#pragma unroll
            for (int e = 0; e < 2; ++e)
                if (writes_angles && key / 2 + e < A) rf.PutD(rf.StartAngle(key / 2 + e), th[e]);
        }
        // the end state turned by the segment's start angles (zero for segment
        // 0, which has the true ones, and for pairs without an angle)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const float rev = static_cast<float>(th[x] * kRevPerTurn);
            const float sn = __builtin_amdgcn_sinf(rev), c = __builtin_amdgcn_cosf(rev);
            const float e0 = cur.end[2 * x], e1 = cur.end[2 * x + 1];
            cur.end[2 * x] = e0 * c - e1 * sn;
            cur.end[2 * x + 1] = e0 * sn + e1 * c;
            th[x] = __builtin_amdgcn_fract(th[x] + cur.dth[x]);
        }
        // the decay in two halves, which keeps its product with S in range
        // where the decay alone is not; a zero state stays zero under any growth
        const float half = __expf(0.5f * cur.decay);
#pragma unroll
        for (int e = 0; e < 4; ++e) S[e] = S[e] == 0.0f ? cur.end[e] : fmaf(half * S[e], half, cur.end[e]);
    }
}

template <int KBW, int NW, int NPW, bool LONG, bool HASZ, int MODE, int PACKED>
void LaunchChunkRows(const Mamba3SisoParams &p, const M3Split &split, hipStream_t stream) {
    using L = M3CLayout<KBW, NW, NPW>;
    const int nseg = MODE == kM3Whole ? 1 : (MODE == kM3State ? (split.maxseg - 1) * (split.ls / split.lf) : split.maxseg);
    constexpr int ROWS = MODE == kM3State ? kStateRows : kRows;
    const int nrb = (p.p + ROWS - 1) / ROWS;
    const long long units = static_cast<long long>(p.batch) * p.nheads * nseg;
    const long long blocks = p.cu_seqlens != nullptr ? XcdSpreadBlocks(units, nrb) : units * nrb;
    if (blocks > 2147483647LL) throw Error(XM_ERR_INVALID_ARGUMENT, "Mamba3SisoFn launch exceeds the grid limit");
    constexpr size_t kLds = MODE == kM3State ? L::kStateBytes : L::kBytes;
    EnsureDynamicLds(reinterpret_cast<const void *>(&Mamba3ChunkKernel<KBW, NW, NPW, LONG, HASZ, MODE, PACKED>), static_cast<int>(kLds));
    if constexpr (MODE == kM3Whole) XM_NOTE_LAUNCH("Mamba3ChunkKernel", {}, KBW, NW, NPW, LONG);
    else XM_NOTE_LAUNCH("Mamba3ChunkKernel", {}, KBW, NW, NPW, LONG, HASZ, MODE);
    hipLaunchKernelGGL((Mamba3ChunkKernel<KBW, NW, NPW, LONG, HASZ, MODE, PACKED>), dim3(static_cast<unsigned>(blocks)), dim3(L::NT),
                       kLds, stream, p, split);
}

template <int KBW, int NW, int NPW, bool LONG, bool HASZ, int MODE>
void LaunchChunkMode(const Mamba3SisoParams &p, const M3Split &split, hipStream_t stream) {
    if constexpr (HASZ && MODE == kM3Whole) LaunchChunkRows<KBW, NW, NPW, LONG, HASZ, MODE, 2>(p, split, stream);
    else if (p.cu_seqlens != nullptr) LaunchChunkRows<KBW, NW, NPW, LONG, HASZ, MODE, 1>(p, split, stream);
    else LaunchChunkRows<KBW, NW, NPW, LONG, HASZ, MODE, 0>(p, split, stream);
}

template <int KBW, int NW, int NPW>
void LaunchSplit(const Mamba3SisoParams &p, const M3Split &split, hipStream_t stream) {
    constexpr int NP = M3CLayout<KBW, NW, NPW>::NP;
    const unsigned bh = static_cast<unsigned>(p.batch) * p.nheads;
    LaunchChunkMode<KBW, NW, NPW, false, false, kM3State>(p, split, stream);
    const int nrb = (p.p + kRows - 1) / kRows, parts = (NP * std::min(kRows, p.p) / 4 + 255) / 256;
    XM_NOTE_LAUNCH("Mamba3SegCombineKernel", {}, );
    hipLaunchKernelGGL(Mamba3SegCombineKernel, dim3(bh * nrb * parts), dim3(256), 0, stream, p, split, NP, parts);
    if (p.Z != nullptr) LaunchChunkMode<KBW, NW, NPW, false, true, kM3Out>(p, split, stream);
    else LaunchChunkMode<KBW, NW, NPW, false, false, kM3Out>(p, split, stream);
}

template <int KBW, int NW, int NPW>
void LaunchChunk(const Mamba3SisoParams &p, bool long_rows, hipStream_t stream) {
    const M3Split none{};
    if (!long_rows) {
        const M3Split split = ChooseSplit(p, M3CLayout<KBW, NW, NPW>::NP);
        if (split.maxseg > 1) return LaunchSplit<KBW, NW, NPW>(p, split, stream);
    }
    if (long_rows && p.Z != nullptr) LaunchChunkMode<KBW, NW, NPW, true, true, kM3Whole>(p, none, stream);
    else if (long_rows) LaunchChunkMode<KBW, NW, NPW, true, false, kM3Whole>(p, none, stream);
    else if (p.Z != nullptr) LaunchChunkMode<KBW, NW, NPW, false, true, kM3Whole>(p, none, stream);
    else LaunchChunkMode<KBW, NW, NPW, false, false, kM3Whole>(p, none, stream);
}

}  // namespace

bool LaunchMamba3SisoChunked(const Mamba3SisoParams &p, void *stream_v) {
    if (GetOverride(kOverrideM3Path) == 1) return false;
    // Buffer descriptors hold 32-bit byte sizes.  The token rows of Q/K,
    // Angles and V/Z/out of one sequence below 2 GiB each: one descriptor per
    // tensor for the whole sequence.  From 2 GiB on: per-chunk descriptors
    // (16 token rows each must stay below 2 GiB).
    const size_t widest = std::max({static_cast<size_t>(p.nheads_qk) * p.n, static_cast<size_t>(p.nheads) * p.a,
                                    static_cast<size_t>(p.nheads) * p.p});
    const size_t row_bytes = widest * sizeof(float);
    if (row_bytes * kC >= (size_t{1} << 31)) return false;
    const bool long_rows = static_cast<size_t>(p.seqlen) * row_bytes >= (size_t{1} << 31);
    hipStream_t stream = static_cast<hipStream_t>(stream_v);
    // headdim_qk padded to 64, 128, 192 or 256 keys
    if (p.n <= 64) LaunchChunk<1, 4, 4>(p, long_rows, stream);
    else if (p.n <= 128) LaunchChunk<2, 4, 8>(p, long_rows, stream);   // 8 product waves: slower (more partials)
    else if (p.n <= 192) LaunchChunk<3, 4, 4>(p, long_rows, stream);
    else if (p.n <= 256) LaunchChunk<4, 4, 4>(p, long_rows, stream);
    else return false;
    XM_LAUNCH_CHECK("Mamba3SisoFn (chunked)");
    return true;
}

}  // namespace xm
