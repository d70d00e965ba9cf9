// The arithmetic of the row quantizers, shared by the row kernels (rowquant.hip)
// and the products that quantize their few rows themselves (gemm_i8.hip).
#pragma once

#include "common.hpp"

namespace xpuint8 {
namespace {

// --------------------------------------------------------------- quantizers
enum QMode : int {
    kRecip = 0,     // ConvRot quantizer: rint(v * (1/s)), s = max(rowmax/127, 1e-30)
                    //   (src/xpuint8.cpp:264-276, 494-498)
    kDivide = 1,    // torch chain: rint(v / s) with IEEE division (ops.py:320-330)
    kPrepare = 2,   // prepare_weight: v rounded to bf16 first, the floor is
                    //   bf16(1e-30), rint(v / s) (ops.py:93-99)
};

__device__ __forceinline__ float row_scale(int mode, float rowmax) {
    if (mode == kPrepare) {
        // bf16(1e-30f) = 0x0DA2 << 16
        return div127_rn(fmaxf(rowmax, __uint_as_float(0x0DA20000u)));
    }
    return fmaxf(div127_rn(rowmax), 1e-30f);
}

// Quantize 16 values: the values themselves unless ROT, in which case the
// rotation is u * dom (dom = 1/16 for the unscaled transform's sums, 1 for the
// scaled one's).
template <bool ROT, int MODE>
__device__ __forceinline__ uint4 quant16(const float (&u)[16], float s, float inv, float dom) {
    if constexpr (MODE == kRecip) {
        // rint(fl(u/16) * inv) == rint(u * fl(inv/16)): both products are exact
        // power-of-two rescalings of the same rounded product.
        const float k = ROT ? inv * dom : inv;
        float a[8], b[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            a[t] = u[t] * k;
            b[t] = u[t + 8] * k;
        }
        const uint2 lo = rint_pack8(a), hi = rint_pack8(b);
        return make_uint4(lo.x, lo.y, hi.x, hi.y);
    } else {
        uint32_t b[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            float x = ROT ? u[t] * dom : u[t];
            if (MODE == kPrepare) x = bf16_round(x);
            b[t] = rint_bits(rint_div(x, s, inv));
        }
        uint4 r;
        r.x = pack4(b[0], b[1], b[2], b[3]);
        r.y = pack4(b[4], b[5], b[6], b[7]);
        r.z = pack4(b[8], b[9], b[10], b[11]);
        r.w = pack4(b[12], b[13], b[14], b[15]);
        return r;
    }
}

// Running max of |u| over 16 raw values.
__device__ __forceinline__ float absmax16(const float (&u)[16], float m) {
#pragma unroll
    for (int t = 0; t < 16; ++t) m = fmaxf(m, fabsf(u[t]));
    return m;
}

// Rotate one lane's register of each of its P groups in place, choosing the
// transform for the whole wave: the unscaled one unless some input of the
// wave is at or above kUnscaledLimit (common.hpp), then the reference's scaled
// one.  Returns dom, the factor from the values left in v to the rotation
// (1/16 or 1), which the callers apply to the row max and in the quantizer;
// both products are exact (a power of two on a value that neither overflows
// nor rounds in the subnormal range).
template <int P>
__device__ __forceinline__ float rotate_groups(float (&v)[P][16], const XlaneSigns& sgn) {
    float mi = 0.f;
#pragma unroll
    for (int p = 0; p < P; ++p) mi = inmax16(v[p], mi);
    if (__builtin_expect(wave_needs_scaled(mi), 0)) {
#pragma unroll
        for (int p = 0; p < P; ++p) hadamard16_scaled(v[p], sgn);
        return 1.0f;
    }
#pragma unroll
    for (int p = 0; p < P; ++p) hadamard16_unscaled(v[p], sgn);
    return 0.0625f;
}

// The row max of the values the quantizer sees, from the max of the rotated
// (or, without ROT, raw) ones: bf16 rounding (kPrepare) is monotone
// non-decreasing, so f(max|u|) == max f(|u|) and one application suffices.
template <int MODE>
__device__ __forceinline__ float finish_max(float x) {
    if (MODE == kPrepare) x = bf16_round(x);
    return x;
}

// s_barrier after this wave's LDS operations have completed, without waiting
// for its outstanding global loads (which __syncthreads() would).  The
// "memory" clobber keeps the compiler from moving memory operations across.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

}  // namespace
}  // namespace xpuint8
