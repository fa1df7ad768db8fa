// HIP error mapping and small device helpers shared by the gfx950 kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "xm_common.h"

#define XM_HIP_CHECK(expr)                                                                         \
    do {                                                                                           \
        hipError_t xm_err_ = (expr);                                                               \
        if (xm_err_ != hipSuccess)                                                                 \
            throw ::xm::Error(XM_ERR_DEVICE, std::string(#expr) + " failed: " + hipGetErrorString(xm_err_)); \
    } while (0)

// Reports a failed launch (reference: XM_CUDA_KERNEL_CHECK, cuda_common.h:27-36).
namespace xm {
// The HIP error this call's launches left on the thread, consumed; hipSuccess
// when there is none, or when the pending error is the one the caller had
// left before the call (ResetLaunches notes it): that one stays for the
// caller's own check.
hipError_t TakeLaunchError();
}  // namespace xm

#define XM_LAUNCH_CHECK(what)                                                                      \
    do {                                                                                           \
        hipError_t xm_err_ = ::xm::TakeLaunchError();                                              \
        if (xm_err_ != hipSuccess)                                                                 \
            throw ::xm::Error(XM_ERR_DEVICE, std::string(what) + " kernel launch failed: " + hipGetErrorString(xm_err_)); \
    } while (0)

namespace xm {

// Raises `kernel`'s dynamic-LDS limit to `bytes` on the current device the
// first time a launch needs it; later launches skip the runtime call.
void EnsureDynamicLds(const void *kernel, int bytes);

constexpr float kLog2eF = 1.4426950408889634f;  // M_LOG2E as float

// Moves `x` across lanes with a DPP control (row-local patterns only).
template <int CTRL>
__device__ __forceinline__ float DppF(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), CTRL, 0xf, 0xf, true));
}

// Sum over the 16 lanes of a DPP row, result in every lane of the row.
// xor 1 and xor 2 (quad_perm), xor 7 (row_half_mirror), xor 8 (row_ror:8)
// span all 16 lanes; each step folds into one v_add_f32_dpp.
__device__ __forceinline__ float RowSum16(float x) {
    x += DppF<0xB1>(x);   // quad_perm [1,0,3,2]
    x += DppF<0x4E>(x);   // quad_perm [2,3,0,1]
    x += DppF<0x141>(x);  // row_half_mirror
    x += DppF<0x128>(x);  // row_ror:8
    return x;
}

// Sum over 64 lanes, result in every lane.  After the row sum every lane of
// row r holds that row's sum; the GFX9 broadcast DPP controls then add row 0
// into row 1 and row 2 into row 3 (row_bcast:15, rows 1 and 3 enabled), and
// lane 31 (rows 0+1) into rows 2 and 3 (row_bcast:31), so lane 63 holds the
// total, which readlane returns to every lane.  No LDS traffic.
__device__ __forceinline__ float WaveSum64(float x) {
    x = RowSum16(x);
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x142, 0xa, 0xf, false));
    x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x143, 0xc, 0xf, false));
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 63));
}

__device__ __forceinline__ double WaveSum64d(double x) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) x += __shfl_xor(x, o);
    return x;
}

// KT consecutive floats of LDS into registers, 16 or 8 bytes at a time.
template <int KT>
__device__ __forceinline__ void LoadKeys(const float *src, float (&x)[KT]) {
    if constexpr (KT % 4 == 0) {
#pragma unroll
        for (int j = 0; j < KT; j += 4) {
            const float4 v = *reinterpret_cast<const float4 *>(src + j);
            x[j] = v.x; x[j + 1] = v.y; x[j + 2] = v.z; x[j + 3] = v.w;
        }
    } else if constexpr (KT % 2 == 0) {
#pragma unroll
        for (int j = 0; j < KT; j += 2) {
            const float2 v = *reinterpret_cast<const float2 *>(src + j);
            x[j] = v.x; x[j + 1] = v.y;
        }
    } else {
#pragma unroll
        for (int j = 0; j < KT; ++j) x[j] = src[j];
    }
}

// Packed sequences: zeros the token rows of `out` ([seqlen][row_floats]) that
// no sequence covers, the part of workgroup wg of nwg (every thread of the
// workgroup calls it).  Sequence b covers [lo_b, hi_b), lo_b = clamp(cu[b]),
// hi_b = clamp(max(cu[b + 1], lo_b)), the ranges the operator kernels use;
// non-decreasing offsets cover exactly [lo_0, hi_{n-1}), so only the rows before
// and after are written (the usual row has none), four floats a thread in one
// stretch each: a workgroup to a row left most threads idle (11872 rows of 64
// floats: 9.4 us, 2.9 so).  Other offsets are checked sequence by sequence
// (malformed input: time linear in n per row).
__device__ __forceinline__ void ZeroPackedGaps(float *out, size_t row_floats, const int64_t *cu, int n, int seqlen,
                                               int wg, int nwg) {
    __shared__ int s_monotone;
    if (threadIdx.x == 0) s_monotone = 1;
    __syncthreads();
    bool mono = true;
    for (int b = threadIdx.x; b < n; b += blockDim.x) mono = mono && cu[b] <= cu[b + 1];
    if (!mono) s_monotone = 0;
    __syncthreads();
    const bool monotone = s_monotone != 0;
    const long long L = seqlen;
    auto clampt = [&](long long x) { return min(max(x, 0LL), L); };
    const long long first = clampt(cu[0]), last = clampt(max(cu[n], first));
    if (monotone) {
        typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));   // out is 4-byte aligned
        const size_t stride = static_cast<size_t>(nwg) * blockDim.x, at = static_cast<size_t>(wg) * blockDim.x + threadIdx.x;
        auto zero = [&](long long t0, long long t1) {   // rows [t0, t1)
            float *dst = out + static_cast<size_t>(t0) * row_floats;
            const size_t count = static_cast<size_t>(t1 - t0) * row_floats;
            for (size_t i = at; i < count / 4; i += stride) reinterpret_cast<f4u *>(dst)[i] = f4u{0.0f, 0.0f, 0.0f, 0.0f};
            if (at < count % 4) dst[count - 1 - at] = 0.0f;
        };
        zero(0, first);
        zero(last, L);
        return;
    }
    for (long long t = wg; t < L; t += nwg) {   // workgroup-uniform
        bool covered = false;
        for (int b = 0; b < n && !covered; ++b) {
            const long long lo = clampt(cu[b]), hi = clampt(max(cu[b + 1], lo));
            covered = t >= lo && t < hi;
        }
        if (!covered)
            for (size_t f = threadIdx.x; f < row_floats; f += blockDim.x) out[static_cast<size_t>(t) * row_floats + f] = 0.0f;
    }
}

// MI355X deals the workgroups of a launch round-robin to its 8 XCDs
// (workgroup x runs on XCD x % 8), and each XCD has its own L2.  This maps
// the hardware index to a logical one under which XCD j owns one contiguous
// range of logical indices, so workgroups that read the same data (adjacent
// logical indices) share an L2 instead of fetching it once per XCD.  It is a
// bijection on [0, n) for any n.
constexpr int kNumXcds = 8;
__device__ __forceinline__ int XcdLocalBlock(int x, int n) {
    const int per = n / kNumXcds, rem = n % kNumXcds;
    const int xcd = x % kNumXcds, slot = x / kNumXcds;
    return xcd < rem ? xcd * (per + 1) + slot : rem * (per + 1) + (xcd - rem) * per + slot;
}
// For packed sequences, whose lengths differ: logical units of `per`
// workgroups each, unit u on XCD u % 8, so that consecutive units (the heads of
// one sequence) spread over the XCDs while a unit's workgroups, which read the
// same data, share an L2.  A contiguous range per XCD (XcdLocalBlock) gives one
// XCD a long sequence's heads, two workgroups to a CU, and leaves others idle.
// The launch has XcdSpreadBlocks(units, per) workgroups; those of a unit >=
// units have nothing to do.
struct XcdUnit {
    int unit, part;   // part: the workgroup within the unit
};
__device__ __forceinline__ XcdUnit XcdSpreadUnit(int x, int per) {
    const int xcd = x % kNumXcds, slot = x / kNumXcds;
    return {slot / per * kNumXcds + xcd, slot % per};
}
inline long long XcdSpreadBlocks(long long units, long long per) {
    return (units + kNumXcds - 1) / kNumXcds * kNumXcds * per;
}

}  // namespace xm
