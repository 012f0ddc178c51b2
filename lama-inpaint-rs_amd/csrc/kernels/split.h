// FP32 products on the bf16 matrix cores.
//
// An f32 value x is taken as three bf16 parts, each the nearest bf16 to what the
// ones before leave,
//     b0 = bf16(x),  b1 = bf16(x - b0),  b2 = bf16(x - b0 - b1).
// Both differences are exact and a part has 8 bits, so b0 + b1 + b2 is x, all 24
// bits of it, with f32's range: no scale is kept, and nothing that an output's
// sum does not read can change it.  A product is then six MFMAs into f32,
//     a x = a0 x0 + a0 x1 + a1 x0 + a1 x1 + a0 x2 + a2 x0
// (a1 x2, a2 x1 and a2 x2, at most 2^-24 of |a x| together, are dropped), each the
// exact product of 8-bit numbers.  v_mfma_f32_32x32x16_bf16 does 16 times the
// products of v_mfma_f32_32x32x2_f32 in the same time, so six of them are 2.7
// times as fast, and the sum is rounded less often: with the small products in
// a sum of their own (mfma_split3), once per 16 channels instead of once per two.
// SpectralTransform, 64 x 64 plane, against f64: 1.9e-7 (f32 MFMAs 3.7e-7);
// whole 512 x 512 pass 1.9e-6 (3.2e-6).
//
// Two f16 halves, hi + lo, would take three MFMAs, but f16's range needs a common
// scale of all values that meet in a sum, in practice of a workgroup's tile:
// values 2^-36 of the tile's largest were then lost, whatever pixel or channel
// they belonged to (whole 512 x 512 pass 3.09 ms, in bf16 parts 3.66).
//
// Below 2^-110 a part of x leaves the range of bf16, whose smallest value is
// 2^-133: the error there is at most 2^-134.  An infinite or NaN x is kept whole
// in b2, with b0 = b1 = 0: the products are then a0 x and zeros, what the f32
// product gives.  Where b0 would round past the largest bf16, it is that one.
#pragma once
#include <type_traits>

#include <hip/hip_runtime.h>

#include "common.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef __bf16 b4 __attribute__((ext_vector_type(4)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));

namespace {

// The bf16 nearest to a and to b as one register, and the two as f32 again.
__device__ __forceinline__ unsigned bf16_pair(float a, float b)
{
    const b2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(unsigned, v);
}
__device__ __forceinline__ float bf16_lo(unsigned p) { return __uint_as_float(p << 16); }
__device__ __forceinline__ float bf16_hi(unsigned p) { return __uint_as_float(p & 0xffff0000u); }

// The three parts of N values, two at a time.  Returns a value that is not
// finite if some x is infinite, NaN or rounds past the largest bf16: the parts
// are then not those of x, and the caller takes them again with ANY = true.
template <bool ANY, int N, class B>
__device__ __forceinline__ float split3(const float (&x)[N], B &p0, B &p1, B &p2)
{
    unsigned q0[N / 2], q1[N / 2], q2[N / 2];
    float check = 0.f;
#pragma unroll
    for (int e = 0; e < N; e += 2) {
        float a = x[e], b = x[e + 1];
        if constexpr (ANY) {
            constexpr float inf = __builtin_inff(), most = 0x1.fep127f;  // the largest bf16
            const bool fa = fabsf(a) < inf, fb = fabsf(b) < inf;
            const float ya = fa ? a : 0.f, yb = fb ? b : 0.f;
            q0[e / 2] = bf16_pair(fminf(fmaxf(ya, -most), most), fminf(fmaxf(yb, -most), most));
            const float ra = ya - bf16_lo(q0[e / 2]), rb = yb - bf16_hi(q0[e / 2]);
            q1[e / 2] = bf16_pair(ra, rb);
            q2[e / 2] = bf16_pair(fa ? ra - bf16_lo(q1[e / 2]) : a, fb ? rb - bf16_hi(q1[e / 2]) : b);
        } else {
            q0[e / 2] = bf16_pair(a, b);
            a -= bf16_lo(q0[e / 2]);
            b -= bf16_hi(q0[e / 2]);
            q1[e / 2] = bf16_pair(a, b);
            a -= bf16_lo(q1[e / 2]);
            b -= bf16_hi(q1[e / 2]);
            q2[e / 2] = bf16_pair(a, b);
            check += a;
            check += b;
        }
    }
    __builtin_memcpy(&p0, q0, sizeof p0);
    __builtin_memcpy(&p1, q1, sizeof p1);
    __builtin_memcpy(&p2, q2, sizeof p2);
    return check;
}

// Whether some lane's check (split3) is not finite; one answer for the wave.
__device__ __forceinline__ bool split3_again(float check) { return __any(!(fabsf(check) < __builtin_inff())); }

// The parts of the six products, the small ones first.
constexpr int SPLIT3_A[6] = {2, 0, 1, 1, 0, 0}, SPLIT3_X[6] = {0, 2, 1, 0, 1, 0};

// c + low += a x as six MFMAs: the largest products into c, the other five, below
// 2^-7 of them, into low (which may be c where registers are short).  Two sums
// round less often, once per 16 channels in the one that counts.
__device__ __forceinline__ void mfma_split3(const b8 &a0, const b8 &a1, const b8 &a2, const b8 &x0, const b8 &x1,
                                            const b8 &x2, f32x16 &c, f32x16 &low)
{
    low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a2, x0, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, x2, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, x1, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a1, x0, low, 0, 0, 0);
    low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, x1, low, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a0, x0, c, 0, 0, 0);
}

}  // namespace
