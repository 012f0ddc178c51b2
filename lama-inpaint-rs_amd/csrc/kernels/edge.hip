// The 7x7 head (model.1, at the end), the stride-2 3x3 convolutions (model.2/3/4)
// and the transposed ones (model.24/27/30) as implicit GEMMs on three bf16 parts
// (split.h).
//
// A workgroup computes 64 output channels x 128 GEMM pixels (TR rows of TC; for
// the transposed convolutions, 128 input positions of one row phase py, both
// column phases: output rows 2m+py).  Wave (wm, wn) owns 32 channels and 64
// pixels, two 32 x 32 accumulators a phase, so that a weight operand feeds 64
// pixels.  K is walked in chunks of 16 channels x T taps.  The chunk's input
// patch, loaded into registers during the chunk before, is split and stored as
// [part][8-channel group][pixel][8], so that an MFMA operand of a tap is one
// 16-byte read a lane over consecutive pixels; a stride-2 patch row keeps its
// even and its odd columns in two runs, so that output pixels' inputs are
// consecutive there too.  The im2col matrix is never formed; reflect padding is
// an index map.  Weights are MFMA operands in operand order ([32 rows][8-channel
// group][tap][part][32][8]) and go straight into registers, three taps ahead (a
// whole chunk ahead, at 234 registers: 981 us against 895 for the stride-2 ones
// at 2048x2048).
//
// What bounds it: the six MFMAs a product (model.2 at 2048x2048: 370 us at the
// bf16 peak; 0.40-0.49 busy), the loads into registers (an L1 access every second
// cycle) and the latency of staging between them, at two workgroups a CU.
// One launch (mean of the three), f32 MFMAs / here, us: stride 2 at 512x512 96 /
// 61, at 2048x2048 1370 / 910; transposed 93 / 65 and 1230 / 806.
#include <hip/hip_runtime.h>

#include "common.h"
#include "split.h"

namespace {

// KIND 0: 3x3 stride 2, reflect padding 1.  KIND 1, 2: row phase py = KIND - 1
// of a k3 s2 p1 op1 transposed convolution, a (1+py) x 2 window from the
// position on, zeros past the bottom and right edge; tap t reads the window
// offset (dy, dx) and feeds column phase px.  py = 0: phase (0,0) at (0,0);
// phase (0,1) at (0,0), (0,1).  py = 1: phase (1,0) at (0,0), (1,0); phase
// (1,1) at (0,0), (0,1), (1,0), (1,1).
template <int KIND, int TR_, int TC_>
struct EdgeCfg {
    static constexpr bool DOWN = KIND == 0;
    static constexpr int PY = DOWN ? 0 : KIND - 1;
    static constexpr int TR = TR_, TC = TC_, S = DOWN ? 2 : 1, T = DOWN ? 9 : PY ? 6 : 3;
    static constexpr int NPH = DOWN ? 1 : 2;  // column phases
    static constexpr int KC = 16;
    static constexpr int PR = DOWN ? 2 * TR + 1 : TR + PY, PC = DOWN ? 2 * TC + 1 : TC + 1;
    static constexpr int HPC = (PC + 1) / 2, PCP = DOWN ? 2 * HPC : PC;  // columns a row holds in LDS
    static constexpr int NP = PR * PC, HT = LAMA_NT / 2, PER = (NP + HT - 1) / HT;
    static constexpr int GS = PR * PCP, PS = 2 * GS, LDS = 3 * PS;  // group and part strides, in b8
    static __device__ __forceinline__ constexpr int col(int c) { return DOWN ? (c & 1) * HPC + (c >> 1) : c; }
    static __device__ __forceinline__ constexpr int dy(int t) { return DOWN ? t / 3 : PY && (t == 1 || t >= 4) ? 1 : 0; }
    static __device__ __forceinline__ constexpr int dx(int t)
    {
        return DOWN ? t % 3 : PY ? (t == 3 || t == 5 ? 1 : 0) : (t == 2 ? 1 : 0);
    }
    static __device__ __forceinline__ constexpr int px(int t) { return DOWN ? 0 : PY ? (t >= 2 ? 1 : 0) : (t >= 1 ? 1 : 0); }
    static_assert(TR * TC == 128, "128 pixels per block");
};

template <class C>
__device__ __forceinline__ void edge_tile(const ConvProblem &P_mem, int b, b8 *xs, float *epl)
{
    const ConvProblem P = P_mem;  // one batch of scalar loads, held across the barriers
    const int mb = b % P.mblocks, t_ = b / P.mblocks;
    const int m0 = mb * 64, y0 = (t_ / P.tiles_x) * C::TR, x0 = (t_ % P.tiles_x) * C::TC;
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, j = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;
    const ConvSeg &sg = P.s0;
    const unsigned cs = (unsigned)sg.cs;
    const int nc = sg.C, ng = (nc + 7) / 8, n = (nc + 15) / 16;
    const LAMA_GLOBAL float *src = gp(sg.src);
    // this wave's 32 channels (rows past M: the last ones again, not stored)
    const LAMA_GLOBAL float *wt = gp(sg.wt) + (long)min((m0 >> 5) + wm, (P.M - 1) >> 5) * 32 * sg.wrow;
    // Items: 8 channels of one patch pixel, channel group ig by the thread's half
    // of the workgroup; byte offsets in a plane, LDS words, and whether the
    // pixel lies in the plane.
    const int ig = wave >> 1, it0 = tid & (C::HT - 1);
    unsigned po[C::PER];
    int pl[C::PER];
    unsigned in = 0;
#pragma unroll
    for (int it = 0; it < C::PER; ++it) {
        const int pix = min(it0 + it * C::HT, C::NP - 1), r = pix / C::PC, c = pix - r * C::PC;
        int iy = y0 * C::S + r, ix = x0 * C::S + c;
        if constexpr (C::DOWN) {
            iy = reflect1(iy - 1, sg.IH);
            ix = reflect1(ix - 1, sg.IW);
            in |= 1u << it;
        } else {
            if (iy < sg.IH && ix < sg.IW) in |= 1u << it;
            iy = min(iy, sg.IH - 1);
            ix = min(ix, sg.IW - 1);
        }
        po[it] = 4u * (unsigned)(iy * sg.IW + ix);
        pl[it] = ig * C::GS + r * C::PCP + C::col(c);
    }
    float d[C::PER][8];
    auto load = [&](int ck) {
        const int c0 = ck * C::KC + 8 * ig;
#pragma unroll
        for (int e = 0; e < 8; ++e) {  // channels past the last one read it again and become zeros
            const LAMA_GLOBAL float *p = src + (long)min(c0 + e, nc - 1) * cs;
#pragma unroll
            for (int it = 0; it < C::PER; ++it) d[it][e] = *at_byte<float>(p, po[it]);
        }
    };
    load(0);
    // lane (g, j): row j of the wave's 32, group 2 ck + g (past the last: the last, against zeros)
    constexpr int RING = 3;
    b8 w0[RING], w1[RING], w2[RING];
    auto load_w = [&](int t, int ck) {
        const unsigned o = (unsigned)(min(2 * ck + g, ng - 1) * (C::T * 1536) + j * 16);
        const LAMA_GLOBAL float *p = wt + t * 384;
        w0[t % RING] = *at_byte<b8>(p, o);
        w1[t % RING] = *at_byte<b8>(p, o + 512u);
        w2[t % RING] = *at_byte<b8>(p, o + 1024u);
    };
#pragma unroll
    for (int t = 0; t < RING; ++t) load_w(t, 0);
    const int ec = min(m0 + (tid & 63), P.M - 1);
    const float ep = tid < 64    ? (P.bias ? gp(P.bias)[ec] : 0.f)
                     : tid < 128 ? (P.scale ? gp(P.scale)[ec] : 1.f)
                                 : (P.scale ? gp(P.shift)[ec] : 0.f);
    f32x16 acc[C::NPH][2], low[C::NPH][2];
#pragma unroll
    for (int p = 0; p < C::NPH; ++p)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[p][h][r] = low[p][h][r] = 0.f;
    // the wave's two runs of 32 pixels
    const b8 *rd[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int p = wn * 64 + h * 32 + j;
        rd[h] = xs + g * C::GS + (p / C::TC) * C::S * C::PCP + p % C::TC;
    }
    auto stage = [&](auto any) {
        float check = 0.f;
#pragma unroll
        for (int it = 0; it < C::PER; ++it) {
            if (it == C::PER - 1 && C::NP % C::HT && it0 + it * C::HT >= C::NP) break;
            b8 *to = xs + pl[it];
            check += split3<decltype(any)::value>(d[it], to[0], to[C::PS], to[2 * C::PS]);
        }
        return check;
    };
    for (int ck = 0; ck < n; ++ck) {
        if (!C::DOWN || (ck + 1) * C::KC > nc) {
#pragma unroll
            for (int it = 0; it < C::PER; ++it) {
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (!(in >> it & 1u) || ck * C::KC + 8 * ig + e >= nc) d[it][e] = 0.f;
            }
        }
        if (ck > 0) __syncthreads();  // every wave is done with the last chunk's operands
        if (split3_again(stage(std::false_type{}))) stage(std::true_type{});
        load(min(ck + 1, n - 1));  // unconditional: the waits then count exactly
        __syncthreads();
        // each tap's operand reads are issued before the tap before it
        b8 x0_[2][2], x1_[2][2], x2_[2][2];
        auto read = [&](int t) {
            const int o = C::dy(t) * C::PCP + C::col(C::dx(t));
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                x0_[t & 1][h] = rd[h][o];
                x1_[t & 1][h] = rd[h][o + C::PS];
                x2_[t & 1][h] = rd[h][o + 2 * C::PS];
            }
        };
        read(0);
#pragma unroll
        for (int t = 0; t < C::T; ++t) {
            if (t + 1 < C::T) read(t + 1);
#pragma unroll
            for (int h = 0; h < 2; ++h)
                mfma_split3(w0[t % RING], w1[t % RING], w2[t % RING], x0_[t & 1][h], x1_[t & 1][h], x2_[t & 1][h], acc[C::px(t)][h],
                            low[C::px(t)][h]);
            if (t + RING < C::T)
                load_w(t + RING, ck);
            else
                load_w(t + RING - C::T, min(ck + 1, n - 1));
            // keep the load here: the scheduler would otherwise sink it below
            // the chunk's last MFMA
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int p = 0; p < C::NPH; ++p)
#pragma unroll
        for (int h = 0; h < 2; ++h) acc[p][h] += low[p][h];
    if (tid < 192) epl[tid] = ep;
    __syncthreads();
    const int row0 = wm * 32 + 4 * g;  // register r: channel m0 + row0 + 8 (r / 4) + r % 4
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int p = wn * 64 + h * 32 + j, y = y0 + p / C::TC, x = x0 + p % C::TC;
        if (y >= P.OH || x >= P.OW) continue;
        LAMA_GLOBAL float *out = gp(P.out) + (long)(m0 + row0) * P.out_cstride +
                                 (C::DOWN ? (long)y * P.outW + x : (long)(2 * y + C::PY) * P.outW + 2 * x);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int rr = 8 * (r >> 2) + (r & 3), cl = row0 + rr;
            if (m0 + cl >= P.M) continue;
            float v[C::NPH];
#pragma unroll
            for (int q = 0; q < C::NPH; ++q) {
                v[q] = acc[q][h][r] + epl[cl];
                v[q] = v[q] * epl[64 + cl] + epl[128 + cl];
                v[q] = P.relu ? fmaxf(v[q], 0.f) : v[q];
            }
            if constexpr (C::DOWN)
                out[(long)rr * P.out_cstride] = v[0];
            else
                *reinterpret_cast<LAMA_GLOBAL float2 *>(out + (long)rr * P.out_cstride) = make_float2(v[0], v[C::NPH - 1]);
        }
    }
}

template <int TR, int TC>
__device__ __forceinline__ void down_body(const ConvProblem *__restrict__ probs, const ProbStarts &ps)
{
    using C = EdgeCfg<0, TR, TC>;
    __shared__ b8 xs[C::LDS];
    __shared__ float epl[192];
    int b = blockIdx.x;
    const int pi = find_problem(ps, b);
    edge_tile<C>(probs[pi], conv_xcd_order(b, probs[pi].nblocks), xs, epl);
}

template <int TR, int TC>
__device__ __forceinline__ void up_body(const ConvProblem *__restrict__ probs, const ProbStarts &ps)
{
    using C0 = EdgeCfg<1, TR, TC>;
    using C1 = EdgeCfg<2, TR, TC>;
    __shared__ b8 xs[C1::LDS];
    __shared__ float epl[192];
    static_assert(C0::LDS <= C1::LDS, "one LDS layout");
    int b = blockIdx.x;
    const int pi = find_problem(ps, b);
    b = conv_xcd_order(b, probs[pi].nblocks);
    if (pi == 0)
        edge_tile<C0>(probs[0], b, xs, epl);
    else
        edge_tile<C1>(probs[1], b, xs, epl);
}

}  // namespace

// 4 x 32-pixel tiles, and 8 x 16 (_q) for planes whose width leaves much of a
// 32-pixel row empty.
#define LAMA_EDGE_KERNEL(NAME, BODY, TR, TC)                                                              \
    extern "C" __global__ void __launch_bounds__(LAMA_NT) __attribute__((amdgpu_waves_per_eu(2)))         \
        NAME(LAMA_CONV_PARAMS)                                                                            \
    {                                                                                                     \
        LAMA_CONV_STARTS;                                                                                 \
        LAMA_STAMP_BEGIN;                                                                                 \
        BODY<TR, TC>(probs, ps);                                                                          \
        LAMA_STAMP_END;                                                                                   \
    }
LAMA_EDGE_KERNEL(lama_conv3x3s2, down_body, 4, 32)
LAMA_EDGE_KERNEL(lama_conv3x3s2_q, down_body, 8, 16)
LAMA_EDGE_KERNEL(lama_convt_rows, up_body, 4, 32)
LAMA_EDGE_KERNEL(lama_convt_rows_q, up_body, 8, 16)
#undef LAMA_EDGE_KERNEL

// model.1: 7x7, reflect pad 3, at most 4 -> 64 channels, BN + ReLU, on the same
// products.  K = 7 rows x 8 columns (the eighth zero) x 4 channels is 14 steps
// of 16, whose weights, 168 registers a lane, are loaded once: a workgroup
// walks tiles of 4 x 32 pixels, blockIdx.x, + gridDim.x, ...  Wave (wm, wn) owns
// 32 channels and two tile rows.  A tile's input patch, loaded during the tile
// before, is split and stored as [part][pixel][4 channels], so that lane group g's operand of a step, columns x + 4 s +
// 2 g and the next one, is two adjacent 8-byte words; two buffers, one barrier
// a tile.
//
// What bounds it: the MFMAs (168 a tile and wave, 287 us of them at 2048x2048)
// and the stores (1.07 GB, 222 us at a copy's rate), half hidden behind each
// other.  F32 MFMAs / here, us: 512x512 67 / 48, 2048x2048 1020 / 621.
namespace {
constexpr int HR = 4, HC = 32, HPR = HR + 6, HPC = HC + 6, HST = 40, HPART = HPR * HST;  // LDS in b4
constexpr int HNP = HPR * HPC, HPER = (HNP + LAMA_NT - 1) / LAMA_NT, HSTEPS = 14;
}  // namespace
extern "C" __global__ void __launch_bounds__(LAMA_NT) __attribute__((amdgpu_waves_per_eu(2)))
lama_conv7x7r(LAMA_CONV_PARAMS)
{
    __shared__ __attribute__((aligned(16))) b4 xs[2 * 3 * HPART];
    __shared__ float epl[192];
    LAMA_STAMP_BEGIN;
    const ConvProblem P = probs[0];
    const ConvSeg &sg = P.s0;
    const int tiles_x = (P.OW + HC - 1) / HC, ntiles = tiles_x * ((P.OH + HR - 1) / HR);
    int t = blockIdx.x;
    if (t >= ntiles) {  // whole workgroup
        LAMA_STAMP_END;
        return;
    }
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, j = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;
    const int nc = sg.C;
    float d[HPER][4];
    auto load = [&](int tile) {
        const int y0 = (tile / tiles_x) * HR, x0 = (tile % tiles_x) * HC;
#pragma unroll
        for (int it = 0; it < HPER; ++it) {
            const int pix = min(tid + it * LAMA_NT, HNP - 1), r = pix / HPC, c = pix - r * HPC;
            const unsigned o = 4u * (unsigned)(reflect1(y0 - 3 + r, sg.IH) * sg.IW + reflect1(x0 - 3 + c, sg.IW));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = *at_byte<float>(gp(sg.src) + (long)min(e, nc - 1) * sg.cs, o);
                d[it][e] = e < nc ? v : 0.f;
            }
        }
    };
    // tile number i of this workgroup, held in d, into its buffer
    auto stage = [&](auto any, int i) {
        b4 *const to = xs + (i & 1) * 3 * HPART;
        float check = 0.f;
#pragma unroll
        for (int it = 0; it < HPER; ++it) {
            const int pix = tid + it * LAMA_NT, r = pix / HPC, c = pix - r * HPC;
            if (HNP % LAMA_NT && it == HPER - 1 && pix >= HNP) break;
            b4 *p = to + r * HST + c;
            check += split3<decltype(any)::value>(d[it], p[0], p[HPART], p[2 * HPART]);
        }
        return check;
    };
    auto stage_any = [&](int i) {
        if (split3_again(stage(std::false_type{}, i))) stage(std::true_type{}, i);
    };
    load(t);
    // weights: [wm][step 2 ky + s][part][g][32][2 columns x 4 channels]
    b8 w0[HSTEPS], w1[HSTEPS], w2[HSTEPS];
    {
        const LAMA_GLOBAL float *p = gp(sg.wt) + (long)min(wm, (P.M - 1) >> 5) * (HSTEPS * 768) + g * 128 + j * 4;
#pragma unroll
        for (int st = 0; st < HSTEPS; ++st) {
            w0[st] = *reinterpret_cast<const LAMA_GLOBAL b8 *>(p + st * 768);
            w1[st] = *reinterpret_cast<const LAMA_GLOBAL b8 *>(p + st * 768 + 256);
            w2[st] = *reinterpret_cast<const LAMA_GLOBAL b8 *>(p + st * 768 + 512);
        }
    }
    if (tid < 192) {
        const int ec = min(tid & 63, P.M - 1);
        epl[tid] = tid < 64    ? (P.bias ? gp(P.bias)[ec] : 0.f)
                   : tid < 128 ? (P.scale ? gp(P.scale)[ec] : 1.f)
                               : (P.scale ? gp(P.shift)[ec] : 0.f);
    }
    stage_any(0);
    const int step = gridDim.x;
    load(min(t + step, ntiles - 1));  // past the last tile: that one again
    const int row0 = wm * 32 + 4 * g;  // register r: channel row0 + 8 (r / 4) + r % 4
    for (int i = 0;; ++i) {
        __syncthreads();
        if (t + step < ntiles) stage_any(i + 1);
        load(min(t + 2 * step, ntiles - 1));
        f32x16 acc[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[h][r] = 0.f;
        const b4 *const rd = xs + (i & 1) * 3 * HPART + 2 * wn * HST + j + 2 * g;
        b8 x[2][3];
        auto read = [&](int u) {  // step u / 2 of tile row u % 2
            const int st = u >> 1;
#pragma unroll
            for (int part = 0; part < 3; ++part) {
                const b4 *p = rd + part * HPART + ((u & 1) + st / 2) * HST + 4 * (st & 1);
                // the eighth column lies outside the window: zeros, as the zero
                // weights it meets would make NaN of an infinity
                const b4 second = (st & 1) && g ? b4{} : p[1];
                x[u & 1][part] = __builtin_shufflevector(p[0], second, 0, 1, 2, 3, 4, 5, 6, 7);
            }
        };
        read(0);
#pragma unroll
        for (int u = 0; u < 2 * HSTEPS; ++u) {
            if (u + 1 < 2 * HSTEPS) read(u + 1);
            const auto &v = x[u & 1];
            mfma_split3(w0[u >> 1], w1[u >> 1], w2[u >> 1], v[0], v[1], v[2], acc[u & 1], acc[u & 1]);
        }
        const int y0 = (t / tiles_x) * HR + 2 * wn, ox = (t % tiles_x) * HC + j;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if (y0 + h >= P.OH || ox >= P.OW) continue;
            LAMA_GLOBAL float *out = gp(P.out) + (long)row0 * P.out_cstride + (long)(y0 + h) * P.outW + ox;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int rr = 8 * (r >> 2) + (r & 3), cl = row0 + rr;
                if (cl >= P.M) continue;
                float v = acc[h][r] + epl[cl];
                v = v * epl[64 + cl] + epl[128 + cl];
                out[(long)rr * P.out_cstride] = P.relu ? fmaxf(v, 0.f) : v;
            }
        }
        t += step;
        if (t >= ntiles) break;
    }
    LAMA_STAMP_END;
}
