// FFC 3x3 convolutions (stride 1, reflect pad 1) as a one-dimensional
// Winograd F(4,3) along x, on three bf16 parts (split.h).
//
// Each output quad (x .. x+3) of a row is computed from the six input columns
// d0..d5 = in[x-1 .. x+4] of each kernel row ky, with the interpolation points
// 0, 1, -1, 2, -2 and infinity (Lavin & Gray, "Fast Algorithms for
// Convolutional Neural Networks", 2016):
//     V = B^T d   (input transform in f32, while the rows are staged in LDS)
//         V0 = 4 d0 - 5 d2 + d4          V3 = -2 d1 - d2 + 2 d3 + d4
//         V1 = -4 (d1 + d2) + d3 + d4    V4 = 2 d1 - d2 - 2 d3 + d4
//         V2 = 4 (d1 - d2) - d3 + d4     V5 = 4 d1 - 5 d3 + d5
//     U = G g     (weight transform in f64, once, by lama_pack_wino)
//         U = (g0/4, -(g0+g1+g2)/6, -(g0-g1+g2)/6, g0/24+g1/12+g2/6, g0/24-g1/12+g2/6, g2)
//     m_u = sum over (ci, ky) of U_u * V_u                   (six GEMMs)
//     out = A^T m (output transform in f32, in the epilogue)
//         out0 = m0 + m1 + m2 + m3 + m4      out2 = m1 + m2 + 4 (m3 + m4)
//         out1 = m1 - m2 + 2 (m3 - m4)       out3 = m1 - m2 + 8 (m3 - m4) + m5
// 6 multiplications per 4 outputs and kernel row instead of 12; the
// transformed values are split.
//
// A workgroup computes 64 output channels x RW rows x 4*NTR pixels (32
// Winograd tiles: RW rows of NTR tiles, NTR = 16, 8 or 4, so 64-, 32- or
// 16-pixel wide blocks).  Wave (wm, wu) owns channels wm*32 .. +32 and the
// positions u = 3*wu .. 3*wu+2 as three 32 x 32 accumulators: GEMM rows are
// output channels, GEMM columns the block's 32 tiles, K = (ci, ky).  K is
// walked in chunks of 16 input channels: the chunk's input rows, loaded into
// registers during the chunk before, are transformed, split and stored as
// [part][8-channel group][row][u][tile][8], so that an MFMA operand is one
// 16-byte read a lane, over consecutive tiles.  Weights are MFMA operands of one
// wave each, in operand order, and go straight into registers, three steps (18
// MFMAs) ahead: nine steps ahead take 72 registers more, which the second sums of
// the products use better, at the same speed (512x512: 3.76 ms with nine and one
// sum, 3.70 with three and two).  In the
// epilogue the two position halves of each channel half swap partial sums of
// the output transform through LDS, so that each wave finishes two of the four
// pixels of every tile.
//
// What bounds it: the bytes into registers (110 KB of weights and 17 KB of inputs
// a chunk and workgroup, 2000 cycles at the L1's 64 bytes a cycle), the MFMAs
// (1728) and the staging's vector instructions (about 1100), which two workgroups
// on a CU overlap only in part: about 5000 cycles a chunk (2048x2048: 0.67 L1
// accesses a cycle, MFMAs 0.34 busy).  Alone, 128 -> 512
// channels, f32 MFMAs / here, us: 64x64 36.6 / 31.7, 128x128 112 / 80, 256x256
// 418 / 296.
#include <hip/hip_runtime.h>

#include "common.h"
#include "split.h"

namespace {

template <int NTR_, bool V4_>
struct W43Cfg {
    // V4: the plane width is a multiple of 4, so each tile's inputs d1..d4 are
    // one aligned 16-byte load (d0 and d5, reflect-mapped at the edges, two
    // scalar ones): three loads per row instead of six
    static constexpr bool V4 = V4_;
    static constexpr int KC = 16;                // input channels per chunk
    static constexpr int NU = 6, KY = 3;         // Winograd positions, kernel rows
    static constexpr int NUW = NU / 2;           // positions per wave
    static constexpr int NS = KY * NUW;          // steps per wave and chunk
    static constexpr int RING = 3;               // steps whose weights are in registers
    static constexpr int NTR = NTR_;             // tiles per output row
    static constexpr int RW = 32 / NTR;          // output rows per block
    static constexpr int TR = RW, TC = 4 * NTR;  // output rows x pixels per block
    static constexpr int IR = TR + 2;            // input rows per block
    static constexpr int NITEM = 4 * IR * NTR;   // (4 channels, row, tile) input items per chunk, at most one a thread
    // LDS, in b8: a row's stride puts the 16 lanes of a read phase, runs of
    // NTR tiles in 16 / NTR rows, on distinct banks
    static constexpr int VRS = NTR == 16 ? 96 : NTR == 8 ? 56 : 28;
    static constexpr int VGS = IR * VRS, VPS = 2 * VGS;  // group and part strides
    static constexpr int V_LDS = 3 * VPS;
    // epilogue exchange: per channel half, two pixels x 16 registers x 64 lanes from each position half
    static constexpr int X_LDS = 2 * 2 * 2 * 16 * 64 / 4;
    static constexpr int LDS = V_LDS > X_LDS ? V_LDS : X_LDS;
    static_assert(NTR * RW == 32, "32 tiles per block");
    static_assert(NITEM <= LAMA_NT, "one item a thread");
};

// d0..d5 of a row to V0..V5.
__device__ __forceinline__ void w43_bt(const float (&d)[6], float (&v)[6])
{
    v[0] = 4.f * d[0] - 5.f * d[2] + d[4];
    v[1] = d[3] + d[4] - 4.f * (d[1] + d[2]);
    v[2] = 4.f * (d[1] - d[2]) - d[3] + d[4];
    v[3] = 2.f * (d[3] - d[1]) - d[2] + d[4];
    v[4] = 2.f * (d[1] - d[3]) - d[2] + d[4];
    v[5] = 4.f * d[1] - 5.f * d[3] + d[5];
}

// One 64-channel x RW-row x 4*NTR-pixel block of problem P (no second segment,
// addends or residual: the FFC's launches store raw partial sums).
template <class C>
__device__ __forceinline__ void w43_tile(const ConvProblem &P_mem, int b, b8 *vs, float *epl)
{
    const ConvProblem P = P_mem;  // one batch of scalar loads, held across the barriers
    // K slice of a split problem: the blocks of slice ks follow those of ks - 1
    int ks = 0;
    if (P.ksplit > 1) {
        const int per = P.mblocks * P.tiles_x * P.tiles_y;
        ks = b / per;
        b -= ks * per;
    }
    // M-block-major: with the XCD-contiguous launch order, an XCD's blocks
    // cover few M blocks (each of whose weights its L2 then holds once)
    const int ntile = P.tiles_x * P.tiles_y, mb = b / ntile, tt = b - mb * ntile;
    const int tx = tt % P.tiles_x, ty = tt / P.tiles_x;
    const int m0 = mb * 64, oy0 = ty * C::TR, ox0 = tx * C::TC;
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, j = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wu = wave & 1;
    const ConvSeg &sg = P.s0;
    const unsigned cs = (unsigned)sg.cs;
    const LAMA_GLOBAL float *src = gp(sg.src);
    // weights: [64 rows][8-channel group][wave][step][part][32][8], 13824 floats a group
    const LAMA_GLOBAL float *wt = gp(sg.wt) + (long)mb * 64 * sg.wrow + wave * (C::NS * 384);
    int nc = sg.C, ng = sg.nchunk / 2;  // channels; packed groups (the pack counts chunks of 4, in pairs)
    if (P.ksplit > 1) {
        const int c0 = ks * P.kchunks * 4;
        src += (long)c0 * cs;
        wt += (long)(c0 / 8) * 13824;
        ng = P.kchunks / 2;
        nc = min(nc - c0, ng * 8);
    }
    const int n = (ng + 1) / 2;
    // This thread's item: channels 4 qc .. + 3 of a chunk at (row ir, tile it).
    // The two quarters of a group are neighbouring lanes, whose 8-byte stores
    // then fill whole 16-byte words.
    const int item = min(tid, C::NITEM - 1);
    const int qc = (item & 1) + 2 * (item / (2 * C::IR * C::NTR));
    const int it = (item >> 1) % C::NTR, ir = (item >> 1) / C::NTR % C::IR;
    // byte offsets of d0..d5 of channel 4 qc from the chunk's first plane
    unsigned po[6];
    {
        const int iy = reflect1(oy0 - 1 + ir, sg.IH);
        const unsigned c0 = 4u * (unsigned)qc * cs;
#pragma unroll
        for (int c = 0; c < 6; ++c) po[c] = 4u * (c0 + (unsigned)(iy * sg.IW + reflect1(ox0 + 4 * it - 1 + c, sg.IW)));
        // d1..d4 in place; a tile past the plane's right edge (outputs
        // dropped) reads the row's last quad instead
        if constexpr (C::V4) po[1] = 4u * (c0 + (unsigned)(iy * sg.IW + min(ox0 + 4 * it, sg.IW - 4)));
    }
    float d[4][6];
    auto load = [&](int ck) {
        const int c0 = ck * C::KC;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const LAMA_GLOBAL float *p = src + (long)(c0 + e) * cs;
            unsigned back = 0;
            if (c0 + C::KC > nc) {  // channels past the last one read it again and become zeros
                const int first = min(c0 + e, nc - 1), want = min(c0 + e + 4 * qc, nc - 1);
                p = src + (long)first * cs;
                back = 4u * (unsigned)(want - first - 4 * qc) * cs;
            }
            if constexpr (C::V4) {
                const float4 m = *at_byte<float4>(p, po[1] + back);
                d[e][0] = *at_byte<float>(p, po[0] + back);
                d[e][1] = m.x;
                d[e][2] = m.y;
                d[e][3] = m.z;
                d[e][4] = m.w;
                d[e][5] = *at_byte<float>(p, po[5] + back);
            } else {
#pragma unroll
                for (int i = 0; i < 6; ++i) d[e][i] = *at_byte<float>(p, po[i] + back);
            }
        }
    };
    load(0);
    // lane (g, j): output channel wm * 32 + j, group 2 ck + g (past the last: the last, against zeros)
    b8 w0[C::RING], w1[C::RING], w2[C::RING];
    auto load_w = [&](int s, int ck) {
        const unsigned o = (unsigned)(min(2 * ck + g, ng - 1) * 55296 + j * 16);
        const LAMA_GLOBAL float *p = wt + s * 384;
        w0[s % C::RING] = *at_byte<b8>(p, o);
        w1[s % C::RING] = *at_byte<b8>(p, o + 512u);
        w2[s % C::RING] = *at_byte<b8>(p, o + 1024u);
    };
#pragma unroll
    for (int s = 0; s < C::RING; ++s) load_w(s, 0);
    const int ec = min(m0 + (tid & 63), P.M - 1);
    const float ep = tid < 64    ? (P.bias ? gp(P.bias)[ec] : 0.f)
                     : tid < 128 ? (P.scale ? gp(P.scale)[ec] : 1.f)
                                 : (P.scale ? gp(P.shift)[ec] : 0.f);
    f32x16 acc[C::NUW], low[C::NUW];
#pragma unroll
    for (int q = 0; q < C::NUW; ++q)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[q][r] = low[q][r] = 0.f;
    // where this item's 4 channels go: V_u at + u * NTR, the parts VPS apart
    b4 *const dst = reinterpret_cast<b4 *>(vs + (qc >> 1) * C::VGS + ir * C::VRS + it) + (qc & 1);
    // the MFMA column's output row and tile within the block
    const b8 *const rd = vs + g * C::VGS + (j / C::NTR) * C::VRS + j % C::NTR + C::NUW * wu * C::NTR;
    auto stage = [&](auto any) {
        float check = 0.f;
        if (C::NITEM < LAMA_NT && tid >= C::NITEM) return check;
        float v[4][6];
#pragma unroll
        for (int e = 0; e < 4; ++e) w43_bt(d[e], v[e]);
#pragma unroll
        for (int u = 0; u < 6; ++u) {
            const float x[4] = {v[0][u], v[1][u], v[2][u], v[3][u]};
            b4 *p = dst + 2 * u * C::NTR;
            check += split3<decltype(any)::value>(x, p[0], p[2 * C::VPS], p[4 * C::VPS]);
        }
        return check;
    };
    for (int ck = 0; ck < n; ++ck) {
        if ((ck + 1) * C::KC > nc) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (ck * C::KC + 4 * qc + e >= nc)
#pragma unroll
                    for (int i = 0; i < 6; ++i) d[e][i] = 0.f;
        }
        if (ck > 0) __syncthreads();  // every wave is done with the last chunk's operands
        if (split3_again(stage(std::false_type{}))) stage(std::true_type{});
        if (ck + 1 < n) load(ck + 1);
        __syncthreads();
        // each step's operand reads are issued before the step before it
        b8 x[2][3];
        auto read = [&](int s) {
            const b8 *p = rd + (s / C::NUW) * C::VRS + (s % C::NUW) * C::NTR;
#pragma unroll
            for (int part = 0; part < 3; ++part) x[s & 1][part] = p[part * C::VPS];
        };
        read(0);
#pragma unroll
        for (int s = 0; s < C::NS; ++s) {
            if (s + 1 < C::NS) read(s + 1);
            const auto &v = x[s & 1];
            mfma_split3(w0[s % C::RING], w1[s % C::RING], w2[s % C::RING], v[0], v[1], v[2], acc[s % C::NUW], low[s % C::NUW]);
            if (s + C::RING < C::NS)
                load_w(s + C::RING, ck);
            else
                load_w(s + C::RING - C::NS, ck + 1);
            // keep the load here: the scheduler would otherwise sink it below
            // the chunk's last MFMA
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int q = 0; q < C::NUW; ++q) acc[q] += low[q];
    // output transform: wave wu = 0 holds m0..m2, wu = 1 holds m3..m5.
    // Partials  p = (m0 + m1 + m2, m1 - m2, m1 + m2, m1 - m2)   (wu = 0)
    //           q = (m3 + m4, 2 (m3 - m4), 4 (m3 + m4), 8 (m3 - m4) + m5)   (wu = 1)
    // and out_i = p_i + q_i; wave wu finishes pixels 2 wu and 2 wu + 1 of each
    // tile, after taking the other half's two partials through LDS.
    float mine[2][16], give[2][16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float a = acc[0][r], b2 = acc[1][r], c = acc[2][r];
        float v[4];
        if (wu == 0) {
            v[0] = a + b2 + c;
            v[1] = b2 - c;
            v[2] = b2 + c;
            v[3] = b2 - c;
        } else {
            v[0] = a + b2;
            v[1] = 2.f * (a - b2);
            v[2] = 4.f * (a + b2);
            v[3] = 8.f * (a - b2) + c;
        }
        mine[0][r] = wu ? v[2] : v[0];
        mine[1][r] = wu ? v[3] : v[1];
        give[0][r] = wu ? v[0] : v[2];
        give[1][r] = wu ? v[1] : v[3];
    }
    // X[wm][from wu][pixel e][r][lane], in the staging buffer
    float *xl = reinterpret_cast<float *>(vs) + wm * 2 * 2 * 16 * 64 + lane;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int r = 0; r < 16; ++r) xl[((wu * 2 + e) * 16 + r) * 64] = give[e][r];
    if (tid < 192) epl[tid] = ep;
    __syncthreads();
    const int oy = oy0 + j / C::NTR, ox = ox0 + 4 * (j % C::NTR) + 2 * wu;
    if (oy >= P.OH || ox >= P.OW) return;
    const bool second = ox + 1 < P.OW;
    const int row0 = wm * 32 + 4 * g;  // register r: channel m0 + row0 + 8 (r / 4) + r % 4
    const long at0 = (long)(m0 + row0) * P.out_cstride + (long)oy * P.outW + ox;
    LAMA_GLOBAL float *out = gp(P.out) + (long)ks * P.out_kstride + at0;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int rr = 8 * (r >> 2) + (r & 3), cl = row0 + rr;
        const long o = (long)rr * P.out_cstride;
        // absent operands are neutral (0, 1, 0)
        float x[2];
#pragma unroll
        for (int e = 0; e < 2; ++e)
            x[e] = mine[e][r] + xl[(((wu ^ 1) * 2 + e) * 16 + r) * 64] + epl[cl];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            x[e] = x[e] * epl[64 + cl] + epl[128 + cl];
            x[e] = P.relu ? fmaxf(x[e], 0.f) : x[e];
        }
        if (m0 + cl >= P.M) continue;
        if constexpr (C::V4) {
            // the width is a multiple of 4 and the rows start at multiples of it: a whole, aligned pair
            *reinterpret_cast<LAMA_GLOBAL float2 *>(out + o) = make_float2(x[0], x[1]);
        } else {
            out[o] = x[0];
            if (second) out[o + 1] = x[1];
        }
    }
}

}  // namespace

// XCD-contiguous launch order: the dispatcher deals workgroups to the eight
// XCDs round-robin (workgroup i to XCD i mod 8), each XCD with its own L2.
// Workgroup i takes block x * q + min(x, r) + i / 8 of the launch's natural
// order (x = i mod 8; the n blocks split as q = n / 8 per XCD, the first
// r = n mod 8 XCDs one more), so that each XCD works through one contiguous
// range: with M-block-major problems that is one or two M blocks' weights
// (0.9 MB each) and one problem's input channels per L2, instead of every
// M block's weights (A: 7.1 MB against a 4 MB L2) or all 384 global input
// planes (B: 6.3 MB) in every L2.
namespace {
__device__ __forceinline__ int wino_xcd_order(int i, int n)
{
    const int x = i & 7, q = n >> 3, r = n & 7;
    return x * q + min(x, r) + (i >> 3);
}
}  // namespace

// Blocks of 2 x 64 (lama_conv3x3w4), 4 x 32 (w4n) or 8 x 16 pixels (w4q);
// problems of a grouped launch are found as in the direct kernels.
#define LAMA_W43_KERNEL(NAME, NTR)                                                          \
    extern "C" __global__ void __launch_bounds__(LAMA_NT)                                   \
        __attribute__((amdgpu_waves_per_eu(LAMA_W43_WAVES))) NAME(LAMA_CONV_PARAMS)         \
    {                                                                                       \
        LAMA_CONV_STARTS;                                                                   \
        LAMA_STAMP_BEGIN;                                                                   \
        using C = W43Cfg<NTR, false>;                                                       \
        using C4 = W43Cfg<NTR, true>;                                                       \
        static_assert(C4::LDS == C::LDS, "one LDS layout");                                 \
        __shared__ b8 vs[C::LDS];                                                           \
        __shared__ float epl[192];                                                          \
        int b = wino_xcd_order(blockIdx.x, gridDim.x);                                      \
        const int pi = find_problem(ps, b);                                                 \
        if (probs[pi].vec_in && (probs[pi].s0.IW & 3) == 0)                                 \
            w43_tile<C4>(probs[pi], b, vs, epl);                                            \
        else                                                                                \
            w43_tile<C>(probs[pi], b, vs, epl);                                             \
        LAMA_STAMP_END;                                                                     \
    }
#ifndef LAMA_W43_WAVES
#define LAMA_W43_WAVES 2
#endif
LAMA_W43_KERNEL(lama_conv3x3w4, 16)
LAMA_W43_KERNEL(lama_conv3x3w4n, 8)
LAMA_W43_KERNEL(lama_conv3x3w4q, 4)
#undef LAMA_W43_KERNEL
