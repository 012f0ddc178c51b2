// The FFCs' weights, packed once when they are loaded: the Winograd transforms of
// the 3x3 convolutions and the pointwise ones as they are.  Each workgroup takes
// one output channel of one matrix, each of its threads an input channel at a
// time, reads its nine taps (its one) and writes their transformed values, in
// three bf16 parts (split.h), into the layout the kernels load as MFMA operands.
//
// The transforms are evaluated in f64 and rounded once to f32, with the same
// terms summed in the same order as the host packer in engine.cpp
// (pack_wino43 / pack_wino42), and each product and sum rounded on its own, as
// on the host: this code object is built with -ffp-contract=fast, under
// which the backend fuses a multiply and an add into one FMA whatever the
// source says, so each product passes through an empty asm statement that
// hides it from that combine.  The packed parts are then identical.
//
// F(4,3) along x: U_u = sum over kx of G[u][kx] w[ky][kx], G for the points
// 0, 1, -1, 2, -2, infinity.  F(2x4, 3x3): U(vy, u) = sum over kx of
// Gx[u][kx] t[vy][kx], t = Gy w (Gy the F(2,3) transform along y, for the
// points 0, 1, -1, infinity).
#include <hip/hip_runtime.h>

#include "common.h"
#include "split.h"

namespace {

// a*x + b*y + c*z, left to right, every operation rounded on its own
__device__ __forceinline__ double dot3(double a, double x, double b, double y, double c, double z)
{
    double p = a * x, q = b * y, r = c * z;
    __asm__ volatile("" : "+v"(p), "+v"(q), "+v"(r));
    return p + q + r;
}

// the three parts of x (split.h), 256 apart
__device__ __forceinline__ void put_parts(LAMA_GLOBAL __bf16 *at, float x)
{
    const float v[2] = {x, 0.f};
    b2 p[3];
    split3<true>(v, p[0], p[1], p[2]);
#pragma unroll
    for (int i = 0; i < 3; ++i) at[256 * i] = p[i][0];
}

// U_u of kernel row ky, u < 6, ky < 3, of one channel pair
__device__ __forceinline__ void transform_w43(const double (&g)[9], float (&v)[6][3])
{
    constexpr double G[6][3] = {{0.25, 0, 0},           {-1.0 / 6, -1.0 / 6, -1.0 / 6}, {-1.0 / 6, 1.0 / 6, -1.0 / 6},
                                {1.0 / 24, 1.0 / 12, 1.0 / 6}, {1.0 / 24, -1.0 / 12, 1.0 / 6}, {0, 0, 1}};
#pragma unroll
    for (int u = 0; u < 6; ++u)
#pragma unroll
        for (int ky = 0; ky < 3; ++ky)
            v[u][ky] = (float)dot3(G[u][0], g[ky * 3], G[u][1], g[ky * 3 + 1], G[u][2], g[ky * 3 + 2]);
}

// [64 rows][8-channel group][wave (wm, u / 3)][step ky * 3 + u % 3][part][32][8]
__device__ __forceinline__ void pack_one_w43(const WinoPackJob &J, int co, int ci, const float (&v)[6][3])
{
    const int mb = co / 64, wm = co % 64 / 32, j = co % 32;
    LAMA_GLOBAL __bf16 *blk = reinterpret_cast<LAMA_GLOBAL __bf16 *>(gp(J.dst)) +
                              ((long)mb * (J.nchunk / 2) + ci / 8) * 27648 + j * 8 + ci % 8;
#pragma unroll
    for (int u = 0; u < 6; ++u)
#pragma unroll
        for (int ky = 0; ky < 3; ++ky) put_parts(blk + ((wm * 2 + u / 3) * 9 + ky * 3 + u % 3) * 768, v[u][ky]);
}

// U(vy, u), vy < 4, u < 6, of one channel pair
__device__ __forceinline__ void transform_w42(const double (&g)[9], float (&v)[4][6])
{
    constexpr double Gx[6][3] = {{0.25, 0, 0},           {-1.0 / 6, -1.0 / 6, -1.0 / 6}, {-1.0 / 6, 1.0 / 6, -1.0 / 6},
                                 {1.0 / 24, 1.0 / 12, 1.0 / 6}, {1.0 / 24, -1.0 / 12, 1.0 / 6}, {0, 0, 1}};
    constexpr double Gy[4][3] = {{1, 0, 0}, {0.5, 0.5, 0.5}, {0.5, -0.5, 0.5}, {0, 0, 1}};
#pragma unroll
    for (int vy = 0; vy < 4; ++vy) {
        double t[3];
#pragma unroll
        for (int kx = 0; kx < 3; ++kx) t[kx] = dot3(Gy[vy][0], g[kx], Gy[vy][1], g[3 + kx], Gy[vy][2], g[6 + kx]);
#pragma unroll
        for (int u = 0; u < 6; ++u) v[vy][u] = (float)dot3(Gx[u][0], t[0], Gx[u][1], t[1], Gx[u][2], t[2]);
    }
}

// [64 rows][8-channel group][wave (wm, vy)][u][part][32][8]
__device__ __forceinline__ void pack_one_w42(const WinoPackJob &J, int co, int ci, const float (&v)[4][6])
{
    const int mb = co / 64, wm = co % 64 / 32, j = co % 32;
    LAMA_GLOBAL __bf16 *blk = reinterpret_cast<LAMA_GLOBAL __bf16 *>(gp(J.dst)) +
                              ((long)mb * (J.nchunk / 2) + ci / 8) * 36864 + wm * 18432 + j * 8 + ci % 8;
#pragma unroll
    for (int i = 0; i < 24; ++i) put_parts(blk + i * 768, v[i / 6][i % 6]);
}

}  // namespace

// [32 rows][8-channel group][part][32][8]
__device__ __forceinline__ void pack_one_pw(const WinoPackJob &J, int co, int ci, float v)
{
    put_parts(reinterpret_cast<LAMA_GLOBAL __bf16 *>(gp(J.dst)) + ((long)(co / 32) * 2 * J.nchunk + ci / 8) * 768 +
                  co % 32 * 8 + ci % 8,
              v);
}

// Grid (x: output channels, y: jobs), 256 threads: a workgroup packs one
// output channel's row; rows past the job's M have nothing to do.
extern "C" __global__ void __launch_bounds__(256) lama_pack_wino(const WinoPackJob *__restrict__ jobs)
{
    const WinoPackJob J = jobs[blockIdx.y];
    const int co = blockIdx.x;
    if (co >= J.M) return;  // whole workgroup
    if (J.kind == 1) {
        for (int ci = threadIdx.x; ci < J.C; ci += 256) pack_one_pw(J, co, ci, gp(J.src0)[(long)co * J.C + ci]);
        return;
    }
    for (int ci = threadIdx.x; ci < J.C; ci += 256) {
        double g[9];
        const LAMA_GLOBAL float *s = ci < J.C0 ? gp(J.src0) + ((long)co * J.C0 + ci) * 9
                                               : gp(J.src1) + ((long)co * (J.C - J.C0) + (ci - J.C0)) * 9;
#pragma unroll
        for (int k = 0; k < 9; ++k) g[k] = (double)s[k];
        if (J.kind == 42) {
            float v[4][6];
            transform_w42(g, v);
            pack_one_w42(J, co, ci, v);
        } else {
            float v[6][3];
            transform_w43(g, v);
            pack_one_w43(J, co, ci, v);
        }
    }
}
