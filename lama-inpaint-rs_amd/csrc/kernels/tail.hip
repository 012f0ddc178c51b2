// model.34 + model.35: 7x7 convolution 64 -> 3 over the ReflectionPad2d(3)
// plane, with bias, then sigmoid (cpu.rs:531-534, 384-388), on three bf16 parts
// (split.h).
//
// Three output channels alone would leave 90% of an MFMA's rows empty, so the
// rows are (channel, kx), 21 of 32: with
//     p[co, kx][y][x'] = sum over (ci, ky) of w[co][ci][ky][kx] in[ci][y + ky][x']
// an output is the sum of seven neighbours, out[co][y][x] = sum over kx of
// p[co, kx][y][x + kx], taken from LDS at the end.  A workgroup computes p for 6
// rows x 64 columns, hence 6 x 58 outputs; wave (rh, ch) owns three rows of 32
// columns, three accumulators.  K is walked in chunks of 16 channels: a chunk's
// 12 x 64 input patch, loaded into registers during the chunk before, is split
// and stored as [part][8-channel group][pixel][8], so that an MFMA operand is one
// 16-byte read a lane; one input row's operand serves up to three output rows
// (ky = 0..6), whose weights the wave holds for the chunk and replaces as soon as
// their last row is done.  Six rows, not eight: 72 KB of LDS, two workgroups a CU
// (84 KB with eight).
//
// What bounds it: the MFMAs and staging (12 x 64 pixels read for 6 x 58 outputs)
// about equally; the input alone is 1.07 GB at 2048x2048, 222 us at a copy's
// rate.  F32 FMAs on the vector units / here, us: 512x512 76 / 55, 2048x2048
// 1180 / 713.
#include <hip/hip_runtime.h>

#include "common.h"
#include "split.h"

namespace {
constexpr int TROWS = LAMA_TAIL_ROWS, TCOLS = LAMA_TAIL_COLS;  // outputs
constexpr int TPR = TROWS + 6, TPC = TCOLS + 6, TNP = TPR * TPC;  // patch
constexpr int THALF = LAMA_NT / 2, TPER = TNP / THALF;         // pixels a thread stages, of one channel group
constexpr int TRW = TROWS / 2;                                 // rows a wave owns
constexpr int TGS = TNP, TPS = 2 * TGS;                        // group and part strides, b8
static_assert(THALF == 2 * TPC && TROWS % 2 == 0 && TROWS <= 8 && TPC == 64, "four waves of TRW rows x 32 columns");
static_assert(TNP % THALF == 0, "whole staging rounds");
static_assert(TROWS * 21 * TPC * 4 <= 3 * TPS * 16, "the sums over (ci, ky) fit in the patch buffer");

}  // namespace

// trunc(clamp(v, 0, 1) * 255 + 0.5) with the product and the sum each
// rounded on its own (main.rs:303-305).  This code object is built with
// -ffp-contract=fast, under which the backend fuses a multiply and an add into
// one FMA (one rounding: a different result for some v) whatever the source
// says; the empty asm statement hides the product from that combine.  NaN
// clamps to 0, as the reference's saturating cast of NaN gives 0.
__device__ __forceinline__ uint8_t composite_u8(float v)
{
    v = fminf(fmaxf(v, 0.f), 1.f);
    float p = v * 255.0f;
    __asm__ volatile("" : "+v"(p));
    return (uint8_t)(int)(p + 0.5f);
}

// U8 = false: the sigmoid plane only.  U8 = true: also the 8-bit composite of
// main.rs:272-307 over the h x w crop -- hole pixels (mask > 0) from the
// network, every other pixel copied from the source bytes.
template <bool U8>
__device__ __forceinline__ void tail_body(const TailArgs *__restrict__ args, int h, int w)
{
    __shared__ b8 xs[3 * TPS];
    const TailArgs A = *args;
    const int H = A.H, W = A.W, nc = A.Cin, n = (nc + 15) / 16;
    const int tiles_x = (W + TCOLS - 1) / TCOLS;
    const int b = conv_xcd_order(blockIdx.x, gridDim.x);
    const int oy0 = (b / tiles_x) * TROWS, ox0 = (b % tiles_x) * TCOLS;
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 5, j = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), rh = wave >> 1, ch = wave & 1;
    const long plane = (long)H * W;
    // This thread's pixels, of channel group ig: column lane of the patch rows 2 it
    // + wave % 2, reflect-mapped (H * W is at most 2^27)
    const int ig = wave >> 1, it0 = tid & (THALF - 1);
    const unsigned col = 4u * (unsigned)reflect1(ox0 - 3 + lane, W);
    int row[TPER];
#pragma unroll
    for (int it = 0; it < TPER; ++it) row[it] = reflect1(oy0 - 3 + 2 * it + (wave & 1), H) * W;
    float d[TPER][8];
    auto load = [&](int ck) {
        const int c0 = ck * 16 + 8 * ig;
#pragma unroll
        for (int e = 0; e < 8; ++e) {  // channels past the last one read it again and become zeros
            const LAMA_GLOBAL float *p = gp(A.src) + (long)min(c0 + e, nc - 1) * plane;
#pragma unroll
            for (int it = 0; it < TPER; ++it) d[it][e] = *at_byte<float>(p + row[it], col);
        }
    };
    load(0);
    // weights: [16-channel chunk][ky][part][8-channel group][32 rows 7 co + kx][8]
    b8 w0[7], w1[7], w2[7];
    auto load_w = [&](int ky, int ck) {
        const LAMA_GLOBAL float *p = gp(A.wt) + (ck * 7 + ky) * 768 + lane * 4;
        w0[ky] = *reinterpret_cast<const LAMA_GLOBAL b8 *>(p);
        w1[ky] = *reinterpret_cast<const LAMA_GLOBAL b8 *>(p + 256);
        w2[ky] = *reinterpret_cast<const LAMA_GLOBAL b8 *>(p + 512);
    };
#pragma unroll
    for (int ky = 0; ky < 7; ++ky) load_w(ky, 0);
    f32x16 acc[TRW];
#pragma unroll
    for (int y = 0; y < TRW; ++y)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[y][r] = 0.f;
    const b8 *const rd = xs + g * TGS + rh * TRW * TPC + ch * 32 + j;
    auto stage = [&](auto any) {
        b8 *const to = xs + ig * TGS + it0;
        float check = 0.f;
#pragma unroll
        for (int it = 0; it < TPER; ++it) {
            b8 *p = to + it * THALF;
            check += split3<decltype(any)::value>(d[it], p[0], p[TPS], p[2 * TPS]);
        }
        return check;
    };
    for (int ck = 0; ck < n; ++ck) {
        if ((ck + 1) * 16 > nc) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (ck * 16 + 8 * ig + e >= nc)
#pragma unroll
                    for (int it = 0; it < TPER; ++it) d[it][e] = 0.f;
        }
        if (ck > 0) __syncthreads();  // every wave is done with the last chunk's operands
        if (split3_again(stage(std::false_type{}))) stage(std::true_type{});
        load(min(ck + 1, n - 1));  // unconditional: the waits then count exactly
        __syncthreads();
        // each input row's operand reads are issued before the row before it
        b8 x[2][3];
        auto read = [&](int r) {
#pragma unroll
            for (int part = 0; part < 3; ++part) x[r & 1][part] = rd[r * TPC + part * TPS];
        };
        read(0);
#pragma unroll
        for (int r = 0; r < TRW + 6; ++r) {
            if (r + 1 < TRW + 6) read(r + 1);
            // the six products of the rows in turn: no MFMA waits for the one before it
#pragma unroll
            for (int i = 0; i < 6; ++i)
#pragma unroll
                for (int y = 0; y < TRW; ++y) {
                    const int ky = r - y;
                    if (ky < 0 || ky > 6) continue;
                    acc[y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        SPLIT3_A[i] == 0 ? w0[ky] : SPLIT3_A[i] == 1 ? w1[ky] : w2[ky], x[r & 1][SPLIT3_X[i]], acc[y], 0, 0, 0);
                }
            if (r >= TRW - 1) load_w(r - (TRW - 1), min(ck + 1, n - 1));
            // keep the load here: the scheduler would otherwise sink it below
            // the chunk's last MFMA
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();  // every wave is done with the operands
    // p[row][7 co + kx][column], in the patch buffer; register r: row 8 (r / 4) + 4 g + r % 4
    float *const ps = reinterpret_cast<float *>(xs);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int i = 8 * (r >> 2) + 4 * g + (r & 3);
        if (i >= 21) continue;
#pragma unroll
        for (int y = 0; y < TRW; ++y) ps[((rh * TRW + y) * 21 + i) * TPC + ch * 32 + j] = acc[y][r];
    }
    __syncthreads();
    const int oy = oy0 + (tid >> 5);
    if ((tid >> 5) >= TROWS || oy >= H) return;
    float bias[3];
#pragma unroll
    for (int co = 0; co < 3; ++co) bias[co] = gp(A.bias)[co];
    float sg[3][2];
    const int px[2] = {tid & 31, (tid & 31) + 32};  // columns of the tile, those from TCOLS on dropped
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        if (px[p] >= TCOLS || ox0 + px[p] >= W) continue;
#pragma unroll
        for (int co = 0; co < 3; ++co) {
            const float *q = ps + ((tid >> 5) * 21 + co * 7) * TPC + px[p];
            float v = 0.f;
#pragma unroll
            for (int kx = 0; kx < 7; ++kx) v += q[kx * TPC + kx];
            v += bias[co];
            sg[co][p] = 1.0f / (1.0f + expf(-v));
            gp(A.out)[co * plane + (long)oy * W + ox0 + px[p]] = sg[co][p];
        }
    }
    if constexpr (U8) {
        if (oy >= h) return;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int ox = ox0 + px[p];
            if (px[p] >= TCOLS || ox >= w) continue;  // w <= W
            const long q = (long)oy * w + ox;
            const bool hole = gp(A.mask)[q] > 0;
#pragma unroll
            for (int co = 0; co < 3; ++co)
                gp(A.out_u8)[3 * q + co] = hole ? composite_u8(sg[co][p]) : gp(A.rgb)[3 * q + co];
        }
    }
}

extern "C" __global__ void __launch_bounds__(LAMA_NT) __attribute__((amdgpu_waves_per_eu(2)))
lama_tail(const TailArgs *__restrict__ args, LAMA_STAMP_PARAMS)
{
    LAMA_STAMP_SCOPE;
    tail_body<false>(args, 0, 0);
}

// The tail with the 8-bit composite of the h x w crop fused in.
extern "C" __global__ void __launch_bounds__(LAMA_NT) __attribute__((amdgpu_waves_per_eu(2)))
lama_tail_u8(const TailArgs *__restrict__ args, int h, int w, int, unsigned long long *__restrict__ stamp)
{
    LAMA_STAMP_SCOPE;
    tail_body<true>(args, h, w);
}
