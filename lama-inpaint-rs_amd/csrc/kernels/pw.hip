// Pointwise (1x1) convolutions over flat planes of N pixels, on three bf16 parts
// (split.h): the SpectralTransform's conv1 and FourierUnit conv (lama_conv1x1*),
// and conv2 with the l2g addend, BN_g, ReLU and the residual fused
// (lama_conv1x1_res*).
//
// A workgroup computes MB output channels x NPX pixels.  Its input strip is
// taken in fills of KC channels: every thread loads PER runs of 8 channels of
// one pixel (a wave's loads are whole 128- or 256-byte lines of a plane,
// whatever its alignment or stride), and each run becomes one 16-byte store of
// each of its three parts into LDS, [part][8-channel group][pixel][8]: the lanes
// of a wave write, and of an MFMA operand read, consecutive 16-byte words.  The
// next fill's loads are in flight meanwhile.  Weights are MFMA operands of one
// wave each, packed in operand order ([32 channels][8-channel group][part][32][8])
// and loaded straight into registers, RING 16-channel steps ahead.  Two waves
// share 32 channels and take every second step each (K halves); their sums meet
// in LDS, and each finishes half the rows.
//
// lama_conv1x1_kh, lama_conv1x1_res_kh: 96 channels x 32 pixels in fills of 192,
// for the planes whose 64 x 64 tiles would give at most two workgroups per CU
// (Engine::tile_variant): what bounds them is the latency of one strip, load to
// store, and the bytes a CU takes through its L1 meanwhile; conv1 at 64 x 64 is
// 256 workgroups, one a CU.  At most 128 registers, so that two six-wave
// workgroups fit a CU and one beside the FFC GEMM's (168: 15.0 us against 11.5 in
// a 512 x 512 pass; K = 384 in one fill, 73 KB of LDS: 14.4).  Alone, f32 MFMAs /
// here: conv1 at 64 x 64 14.0 / 11.3 us, the FU conv 11.2 / 10.2 and 14.4 / 13.9
// at 192 and 384 channels.
// lama_conv1x1, lama_conv1x1_res: 64 channels x 64 pixels in fills of 96, the
// larger planes, where the weights feed twice the pixels and three workgroups a
// CU cover each other's loads (conv1 in a 1024 x 1024 pass 47 us; 96-channel tiles
// of six waves 52).  256 x 256 plane, alone, f32 MFMAs / here: conv1 95 / 69 us,
// the FU conv 95 / 73, conv2 134 / 115.  Nothing is saturated there: MFMAs 0.3
// busy, an L1 access every third cycle.
#include <hip/hip_runtime.h>

#include "common.h"
#include "split.h"

#ifndef LAMA_PW_KC
#define LAMA_PW_KC 96
#endif

namespace {

template <int NPX_, int MW_, int KC_>
struct PwCfg {
    static constexpr int NPX = NPX_, MW = MW_, KC = KC_;  // pixels; waves along M; channels per fill
    static constexpr int WAVES = 2 * MW, NT = 64 * WAVES;
    static constexpr int MB = 32 * MW, NCB = NPX / 32;
    static constexpr int KG = KC / 8, KS = KC / 16;         // groups and 16-channel steps per fill
    static constexpr int WS = KS / 2;                       // steps per wave and fill
    static constexpr int RING = WS % 4 == 0 ? 4 : 3;        // weight steps in registers
    static constexpr int PER = KG * NPX / NT, GPR = NT / NPX;  // runs per thread; groups per round of runs
    static constexpr int GPW = 64 / NPX;                    // groups per wave of a round
    static constexpr int XP = KG * NPX, XL = 3 * XP;        // LDS b8s of one part, of the three
    static_assert(PER * NT == KG * NPX && (NPX == 32 || NPX == 64), "whole runs");
    static_assert(WS % RING == 0, "the ring holds a whole number of laps per fill");
    static_assert(MW * NCB * 16 * 64 * 4 <= XL * 16, "the halves' exchange fits the strip's LDS");
};

// One MB x NPX tile of problem P.
//
// K split (P.ksplit > 1, from the host for small planes whose tiles leave
// most CUs idle): the blocks of slice ks follow those of ks - 1; slice ks
// walks input channels [ks * kchunks * 16, + kchunks * 16) and stores its raw
// partial at out + ks * out_kstride (the host clears bias, BN, ReLU, addends
// and residual; the consumer sums the partials and applies them).
template <class C, bool RES>
__device__ __forceinline__ void pw_tile(const ConvProblem &P_mem, int b, b8 *xs, float *epl)
{
    const ConvProblem P = P_mem;  // one batch of scalar loads, held across the barriers
    int ks = 0;
    if (P.ksplit > 1) {
        const int per = P.mblocks * P.tiles_x;
        ks = b / per;
        b -= ks * per;
    }
    int mb = b % P.mblocks, t = b / P.mblocks;
#if LAMA_PW_XCD
    // XCD-aware order: workgroups are dealt to the eight XCDs round-robin
    // (XCD = blockIdx.x mod 8, here b, the launch's only problem), and each
    // XCD has an L2 of its own; giving all M blocks of pixel strip t to XCD
    // t mod 8 makes each strip travel from HBM into one L2 once, instead of
    // once per M block.  The host opts in by sizing the grid for the strips
    // rounded up to a multiple of 8; blocks of the padding strips return
    // (the whole workgroup, before any barrier).
    if (P.ksplit <= 1 && P.nblocks == (P.tiles_x + 7) / 8 * 8 * P.mblocks) {
        const int j = b >> 3;
        mb = j % P.mblocks;
        t = (j / P.mblocks) * 8 + (b & 7);
        if (t >= P.tiles_x) return;
    }
#endif
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, j = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, kh = wave & 1;
    const int m0 = mb * C::MB, ox0 = t * C::NPX;
    const ConvSeg &sg = P.s0;
    const int N = sg.IH * sg.IW;
    const long cs = sg.cs;
    int nc = sg.C, n16 = sg.nchunk;
    const LAMA_GLOBAL float *src = gp(sg.src);
    // this wave's 32 channels (rows past M: the last ones again, not stored)
    const LAMA_GLOBAL float *wt = gp(sg.wt) + (long)min((m0 >> 5) + wm, (P.M - 1) >> 5) * 32 * sg.wrow;
    if (P.ksplit > 1) {
        const int c0 = ks * P.kchunks * 16;
        src += (long)c0 * cs;
        wt += (long)c0 / 8 * 384;
        n16 = P.kchunks;
        nc = min(nc - c0, n16 * 16);
    }
    const int nf = (n16 + C::KS - 1) / C::KS;
    // Runs: round `it` of a thread is group it * GPR + its wave's share, at
    // its pixel (clamped to the plane).  Addresses are a uniform base and a
    // 32-bit byte offset of the lane (below 2^32: a plane is below 2^24 floats).
    const int px = min(ox0 + (C::NPX == 32 ? j : lane), N - 1);
    const unsigned xoff = 4u * ((unsigned)px + (C::NPX == 32 ? 8u * (unsigned)g * (unsigned)cs : 0u));
    const int wgrp = C::NPX == 32 ? 2 * wave : wave;
    float r[C::PER][8];
    auto load = [&](int f) {
        const int nk = nc - f * C::KC;
        if (min(C::KC, nk) % (8 * C::GPW) == 0) {  // whole runs of every wave; zeros past them
#pragma unroll
            for (int it = 0; it < C::PER; ++it)
                if (8 * (it * C::GPR + wgrp) < nk) {
                    const LAMA_GLOBAL float *p = src + (long)(f * C::KC + 8 * (it * C::GPR + wgrp)) * cs;
#pragma unroll
                    for (int e = 0; e < 8; ++e, p += cs) r[it][e] = *at_byte<float>(p, xoff);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) r[it][e] = 0.f;
                }
        } else {  // a ragged channel count, value by value
#pragma unroll
            for (int it = 0; it < C::PER; ++it)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int c = 8 * (it * C::GPR + wgrp + (C::NPX == 32 ? g : 0)) + e;
                    const float v = src[(long)(f * C::KC + min(c, nk - 1)) * cs + px];
                    r[it][e] = c < nk ? v : 0.f;
                }
        }
    };
    load(0);
    // weights: lane (g, j) takes row j and group 2 k16 + g
    b8 w0[C::RING], w1[C::RING], w2[C::RING];
    const unsigned woff = (unsigned)(g * 1536 + j * 16);
    auto load_w = [&](int sl, int f, int s) {
        const int k16 = min(f * C::KS + 2 * s + kh, n16 - 1);
        const LAMA_GLOBAL float *p = wt + (long)k16 * 768;
        w0[sl] = *at_byte<b8>(p, woff);
        w1[sl] = *at_byte<b8>(p, woff + 512u);
        w2[sl] = *at_byte<b8>(p, woff + 1024u);
    };
#pragma unroll
    for (int s = 0; s < C::RING; ++s) load_w(s, 0, s);
    // per-channel epilogue operands: loaded here, parked in LDS with the first fill
    float ep[3];
    {
        const int c = min(m0 + min(tid, C::MB - 1), P.M - 1);
        ep[0] = P.bias ? gp(P.bias)[c] : 0.f;
        ep[1] = P.scale ? gp(P.scale)[c] : 1.f;
        ep[2] = P.scale ? gp(P.shift)[c] : 0.f;
    }
    f32x16 acc[C::NCB], low[C::NCB];
#pragma unroll
    for (int h = 0; h < C::NCB; ++h)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc[h][q] = low[h][q] = 0.f;
    auto stage = [&](auto any) {
        float check = 0.f;
#pragma unroll
        for (int it = 0; it < C::PER; ++it) {
            b8 *to = xs + tid + it * C::NT;  // [part][group][pixel]
            check += split3<decltype(any)::value>(r[it], to[0], to[C::XP], to[2 * C::XP]);
        }
        return check;
    };
    for (int f = 0; f < nf; ++f) {
        if (f > 0) __syncthreads();  // every wave is done with the last fill's strip
        if (split3_again(stage(std::false_type{}))) stage(std::true_type{});
        if (f == 0 && tid < C::MB)
#pragma unroll
            for (int i = 0; i < 3; ++i) epl[i * C::MB + tid] = ep[i];
        if (f + 1 < nf) load(f + 1);
        __syncthreads();
        // laps of the ring; the steps of a lap past the last channel multiply zeros
#pragma unroll
        for (int lap = 0; lap < C::WS; lap += C::RING) {
            if (f * C::KS + 2 * lap >= n16) break;
#pragma unroll
            for (int i = 0; i < C::RING; ++i) {
                const int s = lap + i;
                const b8 *x = xs + (2 * (2 * s + kh) + g) * C::NPX + j;
#pragma unroll
                for (int h = 0; h < C::NCB; ++h)
                    mfma_split3(w0[i], w1[i], w2[i], x[32 * h], x[32 * h + C::XP], x[32 * h + 2 * C::XP], acc[h],
                                low[h]);
                // this step's registers: the step RING on, here or in the next fill
                if (s + C::RING < C::WS)
                    load_w(i, f, s + C::RING);
                else
                    load_w(i, f + 1, i);
            }
        }
    }
#pragma unroll
    for (int h = 0; h < C::NCB; ++h) acc[h] += low[h];
    // K halves: each of the two waves finishes eight of the 16 register rows,
    // handing the other eight over
    float *ex = reinterpret_cast<float *>(xs) + wm * C::NCB * 16 * 64 + lane;
    __syncthreads();
#pragma unroll
    for (int h = 0; h < C::NCB; ++h)
#pragma unroll
        for (int q = 0; q < 8; ++q) ex[(h * 16 + kh * 8 + q) * 64] = kh ? acc[h][q] : acc[h][8 + q];
    __syncthreads();
#pragma unroll
    for (int h = 0; h < C::NCB; ++h)
#pragma unroll
        for (int q = 0; q < 8; ++q)
            acc[h][q] = (kh ? acc[h][8 + q] : acc[h][q]) + ex[(h * 16 + (kh ^ 1) * 8 + q) * 64];
    constexpr int NQ = 8;
    // Register q: channel row0 + 8 (q / 4) + q % 4 + 4 g.  FULL: all of the wave's
    // 2 NQ channels exist, and an address is a uniform row base and a lane offset.
    const int row0 = m0 + 32 * wm + 16 * kh;
    auto finish = [&](auto full_) {
        constexpr bool FULL = decltype(full_)::value;
        const long ocs = P.out_cstride;
        auto at = [&](auto *base, int q) {
            const int row = row0 + 8 * (q >> 2) + (q & 3);
            return base + (FULL ? (long)row * ocs : (long)min(row + 4 * g, P.M - 1) * ocs);
        };
#pragma unroll
        for (int h = 0; h < C::NCB; ++h) {
            const int opx = ox0 + 32 * h + j;
            const unsigned off = 4u * ((unsigned)min(opx, N - 1) + (FULL ? 4u * (unsigned)g * (unsigned)ocs : 0u));
            float add[NQ], res[NQ];
            (void)add;
            (void)res;
            if constexpr (RES) {
#pragma unroll
                for (int q = 0; q < NQ; ++q) add[q] = res[q] = 0.f;
                if (P.res)
#pragma unroll
                    for (int q = 0; q < NQ; ++q) res[q] = *at_byte<float>(at(gp(P.res), q), off);
                // the addend's K slices, summed in order
                for (int i = 0; i < P.naddend; ++i)
#pragma unroll
                    for (int q = 0; q < NQ; ++q)
                        add[q] += *at_byte<float>(at(gp(P.addend) + i * P.addend_kstride, q), off);
            }
            LAMA_GLOBAL float *out = gp(P.out) + (long)ks * P.out_kstride;
            if (opx >= N) continue;
#pragma unroll
            for (int q = 0; q < NQ; ++q) {
                const int cl = row0 - m0 + 4 * g + 8 * (q >> 2) + (q & 3);
                // absent operands are neutral (0, 1, 0): no branch a value
                float v = acc[h][q] + epl[cl];
                if constexpr (RES) v += add[q];
                v = v * epl[C::MB + cl] + epl[2 * C::MB + cl];
                v = P.relu ? fmaxf(v, 0.f) : v;
                if constexpr (RES) v += res[q];
                if (FULL || m0 + cl < P.M) *at_byte<float>(at(out, q), off) = v;
            }
        }
    };
    if (row0 + 2 * NQ <= P.M)
        finish(std::true_type{});
    else
        finish(std::false_type{});
}

}  // namespace

#define LAMA_PW_KERNEL(NAME, NPX, MW, KC, RES)                                                          \
    extern "C" __global__ void __launch_bounds__((PwCfg<NPX, MW, KC>::NT))                              \
        __attribute__((amdgpu_waves_per_eu(NPX == 64 ? 3 : 4))) NAME(LAMA_CONV_PARAMS)                  \
    {                                                                                                   \
        side_priority();                                                                                \
        LAMA_CONV_STARTS;                                                                               \
        LAMA_STAMP_BEGIN;                                                                               \
        using C = PwCfg<NPX, MW, KC>;                                                                   \
        __shared__ b8 xs[C::XL];                                                                        \
        __shared__ float epl[3 * C::MB];                                                                \
        int b = blockIdx.x;                                                                             \
        const int pi = find_problem(ps, b);                                                             \
        pw_tile<C, RES>(probs[pi], b, xs, epl);                                                         \
        LAMA_STAMP_END;                                                                                 \
    }
LAMA_PW_KERNEL(lama_conv1x1, 64, LAMA_PW_MB / 32, LAMA_PW_KC, false)
LAMA_PW_KERNEL(lama_conv1x1_kh, 32, LAMA_PW_KH_MB / 32, 192, false)
LAMA_PW_KERNEL(lama_conv1x1_res, 64, LAMA_PW_MB / 32, LAMA_PW_KC, true)
LAMA_PW_KERNEL(lama_conv1x1_res_kh, 32, LAMA_PW_KH_MB / 32, 192, true)
#undef LAMA_PW_KERNEL
