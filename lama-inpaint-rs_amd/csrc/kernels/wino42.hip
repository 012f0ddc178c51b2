// FFC 3x3 convolutions (stride 1, reflect pad 1) as a two-dimensional
// Winograd F(2x4, 3x3) on three bf16 parts (split.h): F(2,3) along y (points
// 0, 1, -1, infinity) times the F(4,3) of lama_conv3x3w4 along x.  An output
// tile is 2 rows x 4 pixels, read from input rows r0..r3 x the six columns
// d0..d5 of each:
//     e(0) = r0 - r2   e(1) = r1 + r2   e(2) = r2 - r1   e(3) = r1 - r3   (B_y^T)
//     V(vy, u) = B_x^T e(vy)
//     U(vy, u) = sum over (ky, kx) of G_y[vy][ky] G_x[u][kx] g[ky][kx]
//         G_y = (1, 0, 0; 1/2, 1/2, 1/2; 1/2, -1/2, 1/2; 0, 0, 1)   (f64, lama_pack_wino)
//     m(vy, u) = sum over ci of U(vy, u) V(vy, u)               (24 GEMMs)
//     out(row 0) = A_x^T (m(0) + m(1) + m(2)),  out(row 1) = A_x^T (m(1) - m(2) - m(3))
// 24 multiplications per 8 outputs and input channel: 2/3 of the
// one-dimensional F(4,3)'s, 1/3 of the direct sum's.
//
// A workgroup (8 waves, one on a CU) computes 64 output channels x 32 tiles:
// two row pairs of 16 tiles.  Wave (wm, vy) owns channels wm*32 .. +32 and the
// six positions (vy, 0..5) as six 32 x 32 accumulators (GEMM columns: the
// block's 32 tiles).  K is walked in chunks of 16 channels through two LDS
// buffers, one barrier a chunk: while the MFMAs of a chunk run, the next one,
// in registers, is transformed, split and stored as [part][8-channel group]
// [position][tile][8], position by position between the MFMAs, and the one
// after it is loaded.  A staging thread takes four channels of one tile
// and one vy, so it combines two input rows before the x transform; d0 and d5
// come from the neighbouring lanes (a tile row is a DPP row), so a row costs
// one 16-byte load a lane and one for the halo columns.  Each wave loads its
// own weights in operand order, two positions (12 MFMAs) ahead.  In the epilogue every wave
// applies A_x^T to its six accumulators and parks the four pixels in LDS; each
// wave then finishes four of the 16 register rows of its channel half, both
// output rows, from the four y positions.
//
// What bounds it: the loads into registers (a chunk's 147 KB of weights, 65 KB
// of inputs and their halos, 3300 cycles at 64 bytes a cycle from the CU's L1;
// its MFMAs take 2304), the staging's vector instructions, and, with one
// workgroup on a CU, what comes before its first MFMA and after its last
// (2048x2048: 0.45 L1 accesses a cycle, MFMAs 0.22 busy, waves waiting for 0.67 of
// their time).  Alone, 128 -> 512 channels, f32 MFMAs / here, us: 256x256 378 /
// 312, 128x128 98 / 78.  The small products share the sums of
// the large ones: second sums have no registers.
#include <hip/hip_runtime.h>

#include "common.h"
#include "split.h"

namespace {

template <bool V4_>
struct W42Cfg {
    static constexpr bool V4 = V4_;        // 16-byte input loads and stores (plane width a multiple of 4)
    static constexpr int KC = 16;          // input channels per chunk
    static constexpr int NU = 6, NTR = 16;  // x positions; tiles per row pair
    static constexpr int NT = 512;
    static constexpr int RING = 2;  // positions whose weights are in registers (3 spill: 447 us against 388 in a 2048x2048 pass)
    static constexpr int VGS = 24 * 32, VPS = 2 * VGS, VBS = 3 * VPS;  // group, part and buffer strides, b8
    static constexpr int X_LDS = 8 * 16 * 64;  // epilogue: 16 registers x 64 lanes of four pixels per wave
    static constexpr int LDS = 2 * VBS > X_LDS ? 2 * VBS : X_LDS;  // 16-byte words
    static_assert(NU % RING == 0, "a ring slot holds the same positions in every chunk");
};

// V_u of the six columns e of a row.
template <int U>
__device__ __forceinline__ float w42_bt(const float (&e)[6])
{
    if constexpr (U == 0) return 4.f * e[0] - 5.f * e[2] + e[4];
    if constexpr (U == 1) return e[3] + e[4] - 4.f * (e[1] + e[2]);
    if constexpr (U == 2) return 4.f * (e[1] - e[2]) - e[3] + e[4];
    if constexpr (U == 3) return 2.f * (e[3] - e[1]) - e[2] + e[4];
    if constexpr (U == 4) return 2.f * (e[1] - e[3]) - e[2] + e[4];
    return 4.f * e[1] - 5.f * e[3] + e[5];
}

// One 64-channel x 4-row x 64-pixel block of problem P (no second segment,
// addends or residual: the FFC's launches store raw partial sums).
template <class C>
__device__ __forceinline__ void w42_tile(const ConvProblem &P_mem, int b, b8 *vs, float *epl)
{
    const ConvProblem P = P_mem;  // one batch of scalar loads, held across the barriers
    // K slice of a split problem: the blocks of slice ks follow those of ks - 1
    int ks = 0;
    if (P.ksplit > 1) {
        const int per = P.mblocks * P.tiles_x * P.tiles_y;
        ks = b / per;
        b -= ks * per;
    }
    const int ntile = P.tiles_x * P.tiles_y, mb = b / ntile, tt = b - mb * ntile;
    const int tx = tt % P.tiles_x, ty = tt / P.tiles_x;
    const int m0 = mb * 64, oy0 = ty * 4, ox0 = tx * 64;
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, j = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 2, vy = wave & 3;
    const ConvSeg &sg = P.s0;
    const unsigned cs = (unsigned)sg.cs;
    const LAMA_GLOBAL float *src = gp(sg.src);
    // weights: [64 rows][8-channel group][wave][u][part][32][8], 18432 floats a group
    const LAMA_GLOBAL float *wt = gp(sg.wt) + (long)mb * 64 * sg.wrow + wave * (C::NU * 384);
    int nc = sg.C, ng = sg.nchunk / 2;  // channels; packed groups (the pack counts chunks of 4, in pairs)
    if (P.ksplit > 1) {
        const int c0 = ks * P.kchunks * 4;
        src += (long)c0 * cs;
        wt += (long)(c0 / 8) * 18432;
        ng = P.kchunks / 2;
        nc = min(nc - c0, ng * 8);
    }
    const int n = (ng + 1) / 2;
    // This thread's item: channels 8 (wave / 4) + 4 qh .. + 3 of a chunk, row
    // pair rp, tile it, position row vy.  Lanes qh = 0 and 1 fill the halves of
    // the same 16-byte words.
    const int it = lane & 15, qh = lane >> 4 & 1, rp = lane >> 5;
    const bool edge = C::V4 && ox0 + 4 * it + 4 == sg.IW;  // d5 is past the plane: reflected, d3
    const float sb = vy == 1 ? 1.f : -1.f;
    // byte offsets of d1..d4 (V4: d1) and of the block's halo column on this
    // lane's side in the two rows, from the plane of channel 8 (wave / 4)
    constexpr int ND = C::V4 ? 1 : 4;
    unsigned po[2][ND], ph[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        // e(vy) = r[ra] + sb r[rb]
        const int r = h == 0 ? (vy == 0 ? 0 : vy == 2 ? 2 : 1) : (vy == 2 ? 1 : vy == 3 ? 3 : 2);
        const unsigned row = (unsigned)reflect1(oy0 - 1 + 2 * rp + r, sg.IH) * (unsigned)sg.IW, c0 = 4u * qh * cs;
        ph[h] = 4u * (c0 + row + (unsigned)reflect1(it < 8 ? ox0 - 1 : ox0 + 64, sg.IW));
        // a tile past the plane's right edge (outputs dropped) reads the row's last quad
        if constexpr (C::V4)
            po[h][0] = 4u * (c0 + row + (unsigned)min(ox0 + 4 * it, sg.IW - 4));
        else
#pragma unroll
            for (int c = 0; c < ND; ++c) po[h][c] = 4u * (c0 + row + (unsigned)reflect1(ox0 + 4 * it + c, sg.IW));
    }
    float d[4][2][4], dh[4][2];
    auto load = [&](int ck) {
        const int c0 = ck * C::KC + 8 * wm;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const LAMA_GLOBAL float *p = src + (long)(c0 + c) * cs;
            unsigned back = 0;
            if (c0 + 8 > nc) {  // channels past the last one read it again and become zeros
                const int first = min(c0 + c, nc - 1), want = min(c0 + c + 4 * qh, nc - 1);
                p = src + (long)first * cs;
                back = 4u * (unsigned)(want - first - 4 * qh) * cs;
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if constexpr (C::V4) {
                    const float4 m = *at_byte<float4>(p, po[h][0] + back);
                    d[c][h][0] = m.x;
                    d[c][h][1] = m.y;
                    d[c][h][2] = m.z;
                    d[c][h][3] = m.w;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) d[c][h][i] = *at_byte<float>(p, po[h][i] + back);
                }
                dh[c][h] = *at_byte<float>(p, ph[h] + back);
            }
        }
    };
    float e[4][6];
    auto combine = [&](int ck) {
        const int left = nc - (ck * C::KC + 8 * wm + 4 * qh);  // channels of this item
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int i = 0; i < 4; ++i) e[c][1 + i] = fmaf(sb, d[c][1][i], d[c][0][i]);
            const float halo = fmaf(sb, dh[c][1], dh[c][0]);
            // from the lane before / after; the row's first / last lane keeps the halo
            e[c][0] = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(halo), __float_as_int(e[c][4]), 0x111,
                                                                 0xf, 0xf, false));
            const float r = __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(halo), __float_as_int(e[c][1]),
                                                                       0x101, 0xf, 0xf, false));
            e[c][5] = edge ? e[c][3] : r;
        }
        if ((ck + 1) * C::KC > nc) {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (c >= left)
#pragma unroll
                    for (int i = 0; i < 6; ++i) e[c][i] = 0.f;
        }
    };
    b4 *const dst = reinterpret_cast<b4 *>(vs + wm * C::VGS + vy * (6 * 32) + rp * 16 + it) + qh;
    auto stage = [&](auto u_, auto any, int ck) {
        constexpr int U = decltype(u_)::value;
        const float x[4] = {w42_bt<U>(e[0]), w42_bt<U>(e[1]), w42_bt<U>(e[2]), w42_bt<U>(e[3])};
        b4 *p = dst + 2 * ((ck & 1) * C::VBS + U * 32);
        return split3<decltype(any)::value>(x, p[0], p[2 * C::VPS], p[4 * C::VPS]);
    };
    auto each_u = [&](auto f) {
        f(std::integral_constant<int, 0>{});
        f(std::integral_constant<int, 1>{});
        f(std::integral_constant<int, 2>{});
        f(std::integral_constant<int, 3>{});
        f(std::integral_constant<int, 4>{});
        f(std::integral_constant<int, 5>{});
    };
    load(0);
    // lane (g, j): output channel wm * 32 + j, group 2 ck + g (past the last: the last, against zeros)
    b8 w0[C::RING], w1[C::RING], w2[C::RING];
    auto load_w = [&](int u, int ck) {
        const unsigned o = (unsigned)(min(2 * ck + g, ng - 1) * 73728 + j * 16);
        const LAMA_GLOBAL float *p = wt + u * 384;
        w0[u % C::RING] = *at_byte<b8>(p, o);
        w1[u % C::RING] = *at_byte<b8>(p, o + 512u);
        w2[u % C::RING] = *at_byte<b8>(p, o + 1024u);
    };
#pragma unroll
    for (int u = 0; u < C::RING; ++u) load_w(u, 0);
    const int ec = min(m0 + (tid & 63), P.M - 1);
    const float ep = tid < 64    ? (P.bias ? gp(P.bias)[ec] : 0.f)
                     : tid < 128 ? (P.scale ? gp(P.scale)[ec] : 1.f)
                                 : (P.scale ? gp(P.shift)[ec] : 0.f);
    if (tid < 192) epl[tid] = ep;
    f32x16 acc[C::NU];
#pragma unroll
    for (int u = 0; u < C::NU; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[u][r] = 0.f;
    combine(0);
    load(min(1, n - 1));
    {
        float check = 0.f;
        each_u([&](auto u) { check += stage(u, std::false_type{}, 0); });
        if (split3_again(check)) each_u([&](auto u) { stage(u, std::true_type{}, 0); });
    }
    combine(min(1, n - 1));
    for (int ck = 0; ck < n; ++ck) {
        __syncthreads();  // chunk ck is staged, the other buffer's readers are done
        load(min(ck + 2, n - 1));  // unconditional: the waits then count exactly
        float check = 0.f;
        // each position's operand reads are issued before the position before it
        b8 x[2][3];
        const b8 *const rd = vs + (ck & 1) * C::VBS + g * C::VGS + vy * (6 * 32) + j;
        auto read = [&](int u) {
#pragma unroll
            for (int part = 0; part < 3; ++part) x[u & 1][part] = rd[u * 32 + part * C::VPS];
        };
        read(0);
        each_u([&](auto u_) {
            constexpr int u = decltype(u_)::value;
            if (u + 1 < C::NU) read(u + 1);
            const auto &v = x[u & 1];
            mfma_split3(w0[u % C::RING], w1[u % C::RING], w2[u % C::RING], v[0], v[1], v[2], acc[u], acc[u]);
            load_w((u + C::RING) % C::NU, ck + (u + C::RING) / C::NU);
            // after the last chunk this stages that one again, unread
            check += stage(u_, std::false_type{}, ck + 1);
            // the six MFMAs depend on each other: the staging's instructions
            // go into their waits
#pragma unroll
            for (int i = 0; i < 6; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x2, 7, 0);
            }
            // keep the load here: the scheduler would otherwise sink it below
            // the chunk's last MFMA
            __builtin_amdgcn_sched_barrier(0);
        });
        if (split3_again(check)) each_u([&](auto u) { stage(u, std::true_type{}, ck + 1); });
        combine(min(ck + 2, n - 1));
    }
    __syncthreads();  // every wave has left the K loop: the staging buffers are free
    // A_x^T = (1, 1, 1, 1, 1, 0; 0, 1, -1, 2, -2, 0; 0, 1, 1, 4, 4, 0; 0, 1, -1, 8, -8, 1)
    float4 *const X = reinterpret_cast<float4 *>(vs) + lane;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float p1 = acc[1][r] + acc[2][r], q1 = acc[1][r] - acc[2][r];
        const float p3 = acc[3][r] + acc[4][r], q3 = acc[3][r] - acc[4][r];
        X[(wave * 16 + r) * 64] =
            make_float4(acc[0][r] + p1 + p3, q1 + 2.f * q3, p1 + 4.f * p3, q1 + 8.f * q3 + acc[5][r]);
    }
    __syncthreads();
    const int oy = oy0 + 2 * (j >> 4), ox = ox0 + 4 * (j & 15);
    if (oy >= P.OH || ox >= P.OW) return;
    LAMA_GLOBAL float *out = gp(P.out) + (long)ks * P.out_kstride + (long)oy * P.outW + ox;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // register row r = 4 vy + i: output channel wm * 32 + 8 vy + 4 g + i
        const int r = 4 * vy + i, cl = wm * 32 + 8 * vy + 4 * g + i;
        float4 q[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) q[v] = X[((wm * 4 + v) * 16 + r) * 64];
        if (m0 + cl >= P.M) continue;
        const float bias = epl[cl], mul = epl[64 + cl], add = epl[128 + cl];
        auto fin = [&](float x) {  // absent operands are neutral (0, 1, 0)
            x = (x + bias) * mul + add;
            return P.relu ? fmaxf(x, 0.f) : x;
        };
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            if (oy + y >= P.OH) continue;
            const float x[4] = {y ? q[1].x - q[2].x - q[3].x : q[0].x + q[1].x + q[2].x,
                                y ? q[1].y - q[2].y - q[3].y : q[0].y + q[1].y + q[2].y,
                                y ? q[1].z - q[2].z - q[3].z : q[0].z + q[1].z + q[2].z,
                                y ? q[1].w - q[2].w - q[3].w : q[0].w + q[1].w + q[2].w};
            LAMA_GLOBAL float *o = out + (long)(m0 + cl) * P.out_cstride + (long)y * P.outW;
            if constexpr (C::V4) {
                // the width is a multiple of 4 and the rows start at multiples of it: a whole, aligned quad
                *reinterpret_cast<LAMA_GLOBAL float4 *>(o) = make_float4(fin(x[0]), fin(x[1]), fin(x[2]), fin(x[3]));
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (ox + c < P.OW) o[c] = fin(x[c]);
            }
        }
    }
}

}  // namespace

extern "C" __global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
    lama_conv3x3w42(LAMA_CONV_PARAMS)
{
    LAMA_CONV_STARTS;
    LAMA_STAMP_BEGIN;
    __shared__ b8 vs[W42Cfg<true>::LDS];
    __shared__ float epl[192];
    int b = wino_xcd_order(blockIdx.x, gridDim.x);
    const int pi = find_problem(ps, b);
    if (probs[pi].vec_in && (probs[pi].s0.IW & 3) == 0)
        w42_tile<W42Cfg<true>>(probs[pi], b, vs, epl);
    else
        w42_tile<W42Cfg<false>>(probs[pi], b, vs, epl);
    LAMA_STAMP_END;
}
