// resample.hip -- rppt_resample_gpu (api/rppt_tensor_audio_augmentations.h:310).
//
// Windowed-sinc resampling with the caller's lookup table (RpptResamplingWindow,
// api/rppdefs.h:751-790), following cpu/kernel/resample.cpp:27-146: outEnd = ceil(L*out/in) in
// FP32; outputs in blocks of 256 whose input position starts from the FP64 block base and then
// advances by the FP32 step in->out once per output; taps [ceil(x) - lobes, ceil(x) + lobes)
// clipped to the clip; the window value is the linear interpolation of the table.  For mono
// input the taps go in groups of four with the truncating table lookup, the four partial sums
// are combined as (s0+s2)+(s1+s3), and the leftover taps use the flooring, clamped lookup -- the
// HOST path's exact order, so results are bit-identical to RPP HOST.
//
// Work split: one wave per 256-output block at a time, lane l taking outputs l, l + 64, ... of it.  A
// lane's input position is where the HOST loop's sequence of FP32 additions arrives; block_positions
// gets there without making them (an addition per output, one after another, was nearly half the time).
// For mono sources (and the fused down-mix, whose multi-channel input is reduced to mono first) with at
// most kMaxScale inputs per output, each wave first stages the input span its block reads into LDS.
// When in/out is an integer k, every input position of a block is an integer, so each output whose taps
// are not clipped at the clip's ends reads its 2*lobes taps at the same window offsets -lobes .. lobes-1:
// those window values are looked up once per block and the output is a plain FIR in the HOST
// order (taps in fours, (s0+s2)+(s1+s3), then the leftover taps), bit for bit what the per-tap
// lookups give.
// Any other ratio looks every tap up.  A workgroup keeps the table in LDS as (value, step to the next) pairs
// and takes several block rows of its clip with it; an unclipped output of a table that covers every tap
// (no index to clamp) then costs 10 vector instructions, one 8-byte gather and one input read per tap,
// bound by the gathers' bank conflicts and vector issue.  32 clips of 3-15 s, 44.1 -> 16 kHz: 262 -> 70 us;
// 48 -> 44.1 kHz 648 -> 150 us.
#include "common.hpp"
#include "down_mix_math.hpp"
#include "resample_math.hpp"

#include <algorithm>
#include <cmath>

namespace rppa {
namespace {

constexpr int kThreads = 512;      // general kernel: eight waves share a table
constexpr int kFirThreads = 256;
constexpr int kBlockOut = 256;
// Inputs per output up to which a block's input span is staged.  The spans take 3.4 KB of LDS per wave: 13.4 KB per
// workgroup of the integer-ratio kernel, 27 KB per workgroup of the general one, which with the pairs of a 4,091-entry
// table (33 KB) puts two of its workgroups, 16 waves, on a CU.
constexpr int kMaxScale = 3;
constexpr int kMaxTaps = 64;   // 2 * lobes up to which the span is staged
constexpr int kMaxPairs = 6144;   // table entries up to which the pair table is used (48 KB of LDS)
constexpr int kSpan = kBlockOut * kMaxScale + kMaxTaps + 8;   // staged floats per wave

// LDS written by this wave is read by its other lanes after this (and the other way round)
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// An integer-ratio block (every input position j*k exact): lane l takes outputs j = l + 64 i, so
// consecutive lanes read taps k floats apart (no LDS bank conflicts for odd k) and store
// consecutive outputs.  Clipped outputs at the clip's ends take the per-tap lookups.
template <int NT>
__device__ __forceinline__ void fir_block(const float *spB, const float *wts, const Win &win, float *y, long long ob,
                                          int outEnd, int k, int lobes, int inBlockRounded, int L, int lane)
{
    float wr[NT > 0 ? NT : 1];
    if (NT > 0) {
#pragma unroll
        for (int t = 0; t < NT; t++) wr[t] = wts[t];
    }
    for (int i = 0; i < kBlockOut / kWave; i++) {
        const int j = lane + kWave * i;
        const long long o = ob + j;
        if (o >= outEnd) break;
        const int xc = j * k;
        int loc0 = xc - lobes, loc1 = xc + lobes;
        float acc;
        if (loc0 + inBlockRounded >= 0 && loc1 + inBlockRounded <= L) {
            acc = NT > 0 ? fir_one<NT>(spB + loc0, wr, 0) : fir_one<0>(spB + loc0, wts, 2 * lobes);
        } else {
            if (loc0 + inBlockRounded < 0) loc0 = -inBlockRounded;
            if (loc1 + inBlockRounded > L) loc1 = L - inBlockRounded;
            acc = resample_one([&](int li) { return spB[li]; }, win, static_cast<float>(xc), loc0, loc1);
        }
        y[o] = acc;
    }
}

// Input positions of outputs lane, lane + 64, lane + 128, lane + 192 of a block: the values the FP32
// sequence x(0) = x0, x(n + 1) = x(n) + step reaches.  Inside one binade every addition after the first
// adds the same multiple of its ulp (the first may round a tie to the even neighbour; from an even value
// every later tie goes the same way), so a run of them is one exact multiply-add; only the additions that
// enter a binade are made.  Some ten runs cover a block.
__device__ __forceinline__ void block_positions(float x0, float step, int lane, float (&pos)[kBlockOut / kWave])
{
    float x = x0;
#pragma unroll
    for (int u = 0; u < kBlockOut / kWave; u++) pos[u] = x0;
    for (int i = 0; i < kBlockOut;) {
        // x = x(i); y, z follow; top: the end of x's binade (0 for a zero or subnormal x)
        const unsigned e = __float_as_uint(x) & 0x7f800000u;
        const float top = e ? __uint_as_float(e + 0x00800000u) : 0.0f;
        const float y = x + step, z = y + step, d = z - y;
        int m = -1;                          // y .. y + m d lie in x's binade
        if (y < top) {
            m = 0;
            if (z < top) {
                m = d > 0.0f ? static_cast<int>(fminf((top - y) / d, static_cast<float>(kBlockOut))) : kBlockOut;
                if (d > 0.0f && fmaf(static_cast<float>(m), d, y) >= top) m--;
            }
        }
#pragma unroll
        for (int u = 0; u < kBlockOut / kWave; u++) {
            const int j = lane + u * kWave - i;
            if (j == 0) pos[u] = x;
            else if (j >= 1 && j <= m + 1) pos[u] = fmaf(static_cast<float>(j - 1), d, y);
        }
        x = m < 0 ? y : fmaf(static_cast<float>(m), d, y) + step;
        i += m + 2;
    }
}

// One unclipped output: taps x[0 .. 2 lobes) at window positions p, p + 1, ... in the HOST order, the table as
// pairs; every index lies inside the table and 2 lobes is a multiple of four.
template <int GROUPS>
__device__ __forceinline__ float interp_one(const float *x, const float2 *pairs, float scale, float center, float p,
                                            int groups)
{
    float p0 = p + 0.f, p1 = p + 1.f, p2 = p + 2.f, p3 = p + 3.f;
    float a0 = 0.f, a1 = 0.f, a2 = 0.f, a3 = 0.f;
    auto tap = [&](float q, float in) {
        const float loc = q * scale + center;
        const float2 t = pairs[static_cast<unsigned>(loc)];
        return in * (t.x + __builtin_amdgcn_fractf(loc) * t.y);   // fract: loc - floor(loc), exact
    };
#pragma unroll
    for (int g = 0; g < (GROUPS > 0 ? GROUPS : groups); g++) {
        a0 = a0 + tap(p0, x[4 * g]);
        a1 = a1 + tap(p1, x[4 * g + 1]);
        a2 = a2 + tap(p2, x[4 * g + 2]);
        a3 = a3 + tap(p3, x[4 * g + 3]);
        p0 = p0 + 4.0f; p1 = p1 + 4.0f; p2 = p2 + 4.0f; p3 = p3 + 4.0f;
    }
    return (a0 + a2) + (a1 + a3);
}

// One clip of a launch, and how its outputs are computed.
template <bool DMIX>
struct Clip {
    const float *x;
    float *y;
    int C, CO, L, outEnd, s0, spanLen;
    int kInt;          // in / out where it is an integer the FIR kernel takes, else 0
    float dw, ir, orr;
    double scale;
    bool staged;

    __device__ __forceinline__ Clip(int b, const float *src, uint32_t srcStride, float *dst, uint32_t dstStride,
                                    const float *inRates, const float *outRates, const int *dims, int lobes, int normalize,
                                    float inRateAll, float outRateAll)
    {
        C = max(dims[2 * b + 1], 1);
        L = min(dims[2 * b], static_cast<int>(srcStride / C));
        CO = DMIX ? 1 : C;                                     // output channels
        ir = inRates ? inRates[b] : inRateAll;
        orr = outRates ? outRates[b] : outRateAll;
        x = src + static_cast<size_t>(b) * srcStride;
        y = dst + static_cast<size_t>(b) * dstStride;
        dw = DMIX ? down_mix_weight(C, normalize) : 1.0f;
        outEnd = static_cast<int>(ceilf(static_cast<float>(L) * orr / ir));
        outEnd = min(outEnd, static_cast<int>(dstStride / CO));
        // (the FP64 quotient of two FP32 rates is an integer k only where k times the one is the other)
        const bool mono = DMIX || C == 1, shortWin = 2 * lobes <= kMaxTaps;
        kInt = !mono || !shortWin ? 0 : (ir == 2.0f * orr ? 2 : (static_cast<double>(ir) == 3.0 * orr ? 3 : 0));
        static_assert(kMaxScale == 3, "the integer ratios");
        // staged span of the block at output ob: inputs from int(ob * scale) + s0 on, spanLen of them (zero
        // outside the clip, never read there); the float input positions drift from the exact ones by far
        // less than the two-sample margins
        s0 = -lobes - 2;
        if (kInt) {
            spanLen = min(kSpan, kBlockOut * kInt + 2 * lobes + 4);
        } else {
            scale = static_cast<double>(ir) / orr;
            staged = mono && scale <= kMaxScale && shortWin;
            spanLen = min(kSpan, static_cast<int>(ceil(kBlockOut * scale)) + 2 * lobes + 4);
        }
    }
    __device__ __forceinline__ float sample(int t) const
    {
        return DMIX ? down_mix_sample(x + static_cast<size_t>(t) * C, C, dw) : x[t];
    }
    // The span from input `at` on to LDS, the wave's loads all issued before any is used (mono and stereo; other
    // channel counts down-mix sample by sample).
    __device__ __forceinline__ void stage(float *sp, int at, int lane) const
    {
        constexpr int kU = (kSpan + kWave - 1) / kWave;
        const bool stereo = DMIX && C == 2 && (reinterpret_cast<uintptr_t>(x) & 7) == 0;   // 8-byte stereo loads
        if (C == 1 || stereo) {
            float v[kU][2];
#pragma unroll
            for (int u = 0; u < kU; u++) {
                const int t = min(max(at + lane + u * kWave, 0), L - 1);
                if (stereo) {
                    const float2 p2 = *reinterpret_cast<const float2 *>(x + 2 * static_cast<size_t>(t));
                    v[u][0] = p2.x;
                    v[u][1] = p2.y;
                } else {
                    v[u][0] = x[t];
                    v[u][1] = 0.0f;
                }
            }
#pragma unroll
            for (int u = 0; u < kU; u++) {
                const int j = lane + u * kWave, t = at + j;
                if (j < spanLen) sp[j] = (t >= 0 && t < L) ? (stereo ? down_mix_sample(v[u], 2, dw) : v[u][0]) : 0.0f;
            }
        } else {
            for (int j = lane; j < spanLen; j += kWave) {
                const int t = at + j;
                sp[j] = (t >= 0 && t < L) ? sample(t) : 0.0f;
            }
        }
    }
};

// DMIX (both kernels): the source is interleaved multi-channel and is down-mixed (HOST order) before
// resampling; the output is mono.  Otherwise the drop-in resample: mono, or channels resampled independently.

// The clips of an integer ratio: one block row per workgroup, no table in LDS, so that many are in flight (HBM-bound).
template <bool DMIX>
__global__ void __launch_bounds__(kFirThreads)
resample_fir_kernel(const float *__restrict__ src, uint32_t srcStride, float *__restrict__ dst, uint32_t dstStride,
                    const float *__restrict__ inRates, const float *__restrict__ outRates, const int *__restrict__ dims,
                    float wScale, float wCenter, int lobes, int lookupSize, const float *__restrict__ lutG, int normalize,
                    float inRateAll, float outRateAll)
{
    __shared__ float wts[kMaxTaps];                        // taps of an unclipped output
    __shared__ float span[kFirThreads / kWave][kSpan];
    const Clip<DMIX> c(blockIdx.y, src, srcStride, dst, dstStride, inRates, outRates, dims, lobes, normalize, inRateAll,
                       outRateAll);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long long row = static_cast<long long>(blockIdx.x) * (kFirThreads / kWave) * kBlockOut, ob = row + wave * kBlockOut;
    if (!c.kInt || row >= c.outEnd) return;
    const int inBlock = static_cast<int>(ob) * c.kInt;     // input of the wave's first output
    if (ob < c.outEnd) c.stage(span[wave], inBlock + c.s0, lane);
    const Win win{lutG, wScale, wCenter, lookupSize};
    const int nGroups = (2 * lobes) / 4;
    if (threadIdx.x < 2 * lobes) {
        const float p = static_cast<float>(static_cast<int>(threadIdx.x) - lobes);
        wts[threadIdx.x] = threadIdx.x < 4 * nGroups ? win.trunc_lookup(p) : win.floor_lookup(p);
    }
    __syncthreads();
    if (ob >= c.outEnd) return;
    const float *spB = span[wave] - c.s0;                  // spB[li] = input inBlock + li
    if (lobes == 16) fir_block<32>(spB, wts, win, c.y, ob, c.outEnd, c.kInt, lobes, inBlock, c.L, lane);
    else fir_block<0>(spB, wts, win, c.y, ob, c.outEnd, c.kInt, lobes, inBlock, c.L, lane);
}

// Every other clip.  PAIRS: the LDS table holds (value, step) pairs.
template <bool DMIX, bool PAIRS>
__global__ void __launch_bounds__(kThreads)
resample_kernel(const float *__restrict__ src, uint32_t srcStride, float *__restrict__ dst, uint32_t dstStride,
                const float *__restrict__ inRates, const float *__restrict__ outRates, const int *__restrict__ dims,
                float wScale, float wCenter, int lobes, int lookupSize, const float *__restrict__ lutG, int normalize,
                float inRateAll, float outRateAll)
{
    extern __shared__ __attribute__((aligned(16))) float lds[];
    float *lut = lds;
    float2 *pairs = reinterpret_cast<float2 *>(lds);
    float *span = lds + (PAIRS ? 2 : 1) * ((lookupSize + 3) / 4 * 4);   // [wave][kSpan] staged input
    const Clip<DMIX> c(blockIdx.y, src, srcStride, dst, dstStride, inRates, outRates, dims, lobes, normalize, inRateAll,
                       outRateAll);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    constexpr int kRowOut = kThreads / kWave * kBlockOut;  // outputs of one block row
    const long long rowStep = static_cast<long long>(gridDim.x) * kRowOut;
    long long row = static_cast<long long>(blockIdx.x) * kRowOut;
    if (c.kInt) return;
    if (c.ir == c.orr) {  // no resampling: a copy of L*C samples (or of the L down-mixed samples)
        const long long n = min(static_cast<long long>(c.L), static_cast<long long>(dstStride / c.CO)) * c.CO;
        for (; row * c.CO < n; row += rowStep)
            for (long long i = row * c.CO + threadIdx.x; i < min(n, (row + kRowOut) * c.CO); i += kThreads)
                c.y[i] = DMIX ? c.sample(static_cast<int>(i)) : c.x[i];
        return;
    }
    if (row >= c.outEnd) return;
    // the pair form: every tap p in [-lobes, lobes) of an unclipped output finds its entry without clamping
    const float first = static_cast<float>(-lobes) * wScale + wCenter, last = static_cast<float>(lobes) * wScale + wCenter;
    const bool whole = PAIRS && c.staged && 2 * lobes % 4 == 0 && first >= 0.0f && last >= 0.0f &&
                       first < static_cast<float>(lookupSize - 1) && last < static_cast<float>(lookupSize - 1);
    if (whole) {
        for (int i = threadIdx.x; i < lookupSize - 1; i += kThreads) {
            const float cur = lutG[i], nxt = lutG[i + 1];
            pairs[i] = make_float2(cur, nxt - cur);
        }
    } else {
        for (int i = threadIdx.x; i < lookupSize; i += kThreads) lut[i] = lutG[i];
    }
    // the table for the other lookups, each with the address space of its own (one pointer to either would make
    // every lookup a flat load: 8 clips of 1-5 s at 44.1 -> 16 kHz with 40 lobes 145 us, 58 this way)
    const Win winG{lutG, wScale, wCenter, lookupSize}, win{lut, wScale, wCenter, lookupSize};
    __syncthreads();                                       // the table; the spans are each wave's own
    float *sp = span + wave * kSpan;
    const float *spB = sp - c.s0;                          // spB[li] = input inBlock + li of the staged block
    const int nGroups = (2 * lobes) / 4;
    for (; row < c.outEnd; row += rowStep) {
        const long long ob = row + wave * kBlockOut;
        if (ob >= c.outEnd) return;
        const double inBlockRaw = static_cast<double>(ob) * c.scale;
        const int inBlock = static_cast<int>(inBlockRaw);
        if (c.staged) {
            wave_lds_sync();
            c.stage(sp, inBlock + c.s0, lane);
            wave_lds_sync();
        }
        float pos[kBlockOut / kWave];
        block_positions(static_cast<float>(inBlockRaw - inBlock), static_cast<float>(c.scale), lane, pos);
#pragma unroll
        for (int i = 0; i < kBlockOut / kWave; i++) {
            const long long o = ob + lane + i * kWave;
            if (o >= c.outEnd) break;
            const float inPos = pos[i];
            const int xc = static_cast<int>(ceilf(inPos));
            int loc0 = xc - lobes, loc1 = xc + lobes;
            if (whole && loc0 + inBlock >= 0 && loc1 + inBlock <= c.L) {
                const float p = static_cast<float>(loc0) - inPos;
                c.y[o] = lobes == 16 ? interp_one<8>(spB + loc0, pairs, wScale, wCenter, p, 8)
                                     : interp_one<0>(spB + loc0, pairs, wScale, wCenter, p, nGroups);
                continue;
            }
            if (loc0 + inBlock < 0) loc0 = -inBlock;
            if (loc1 + inBlock > c.L) loc1 = c.L - inBlock;
            if (whole) {
                c.y[o] = resample_one([&](int li) { return spB[li]; }, winG, inPos, loc0, loc1);
            } else if (c.staged) {
                c.y[o] = resample_one([&](int li) { return spB[li]; }, win, inPos, loc0, loc1);
            } else if (DMIX || c.C == 1) {
                c.y[o] = resample_one([&](int li) { return c.sample(inBlock + li); }, win, inPos, loc0, loc1);
            } else {
                float acc[16];
                const int Cc = min(c.C, 16);
                for (int ch = 0; ch < 16; ch++) acc[ch] = 0.0f;
                float xx = static_cast<float>(loc0) - inPos;
                for (int li = loc0; li < loc1; li++, xx += 1.0f) {
                    const float w = win.floor_lookup(xx);
#pragma unroll
                    for (int ch = 0; ch < 16; ch++)
                        if (ch < Cc) {
                            float q = c.x[(static_cast<size_t>(inBlock) + li) * c.C + ch] * w;
                            acc[ch] = acc[ch] + q;
                        }
                }
#pragma unroll
                for (int ch = 0; ch < 16; ch++)
                    if (ch < Cc) c.y[o * c.C + ch] = acc[ch];
            }
        }
    }
}

// The launches over [B] clips: the integer-ratio kernel and the general one, each leaving the other's clips at
// once (with rates in device memory the host cannot tell).  An idle launch costs 1.4 us on one clip and 4.7 us in the FIR's
// 7,328 workgroups on the 32 clips above; the general kernel's 3,680 leave in 3.6-6.5 us.  One kernel for both ran the
// FIR at the table's occupancy: 29 us on those clips at 48 -> 16 kHz, 24.7 split, 23 with the FIR alone.  Rates
// the host knows (inRates null) launch the one that applies.
template <bool DMIX>
hipError_t resample_launch(hipStream_t st, const float *src, uint32_t srcStride, float *dst, uint32_t dstStride, unsigned B,
                           const float *inRates, const float *outRates, const int *dims, const RpptResamplingWindow &w,
                           int normalize, float inRate, float outRate)
{
    const double ratio = inRates ? 0.0 : static_cast<double>(inRate) / outRate;
    const bool canFir = 2 * w.lobes <= kMaxTaps, wholeRatio = ratio > 1.0 && ratio <= kMaxScale && ratio == std::floor(ratio);
    if (canFir && (inRates || wholeRatio)) {
        const dim3 grid(std::max(1u, ceil_div(dstStride, kBlockOut * (kFirThreads / kWave))), B);
        hipLaunchKernelGGL(resample_fir_kernel<DMIX>, grid, dim3(kFirThreads), 0, st, src, srcStride, dst, dstStride, inRates,
                           outRates, dims, w.scale, w.center, w.lobes, w.lookupSize, w.lookupPinned, normalize, inRate, outRate);
    }
    if (inRates || !(canFir && wholeRatio)) {
        const bool pairTable = w.lookupSize <= kMaxPairs;
        const size_t bytes = sizeof(float) * ((pairTable ? 2 : 1) * ((w.lookupSize + 3) / 4 * 4) + (kThreads / kWave) * kSpan);
        // a workgroup takes further block rows of its clip with its table where there are more rows than
        // about eight workgroups per CU
        const unsigned rows = ceil_div(dstStride, kBlockOut * (kThreads / kWave));
        const unsigned per = std::max<unsigned>(1, static_cast<unsigned>(static_cast<size_t>(rows) * B / 2048));
        const dim3 grid(std::max(1u, (rows + per - 1) / per), B);
        auto kernel = pairTable ? &resample_kernel<DMIX, true> : &resample_kernel<DMIX, false>;
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(bytes));
        hipLaunchKernelGGL(kernel, grid, dim3(kThreads), bytes, st, src, srcStride, dst, dstStride, inRates, outRates, dims,
                           w.scale, w.center, w.lobes, w.lookupSize, w.lookupPinned, normalize, inRate, outRate);
    }
    return hipGetLastError();
}

// Each clip's resampled length, ceil(samples * outRate / inRate) in FP32 as the resample kernel
// computes its output count.
__global__ void resampled_length_kernel(const int *__restrict__ dims, uint32_t srcStride, float inRate, float outRate,
                                        int B, int *__restrict__ lengths)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= B) return;
    const int C = max(dims[2 * b + 1], 1);
    const int L = max(min(dims[2 * b], static_cast<int>(srcStride / C)), 0);
    const float lf = static_cast<float>(L) * outRate;
    lengths[b] = static_cast<int>(ceilf(lf / inRate));
}

}  // namespace

hipError_t down_mix_resample_launch(hipStream_t st, const float *src, uint32_t srcStride, float *dst,
                                    uint32_t dstStride, unsigned B, const int *dims, float inRate, float outRate,
                                    const RpptResamplingWindow &w, int normalize, int *lengths)
{
    const hipError_t e = resample_launch<true>(st, src, srcStride, dst, dstStride, B, nullptr, nullptr, dims, w, normalize,
                                               inRate, outRate);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(resampled_length_kernel, dim3(ceil_div(B, 256u)), dim3(256), 0, st, dims, srcStride, inRate,
                       outRate, static_cast<int>(B), lengths);
    return hipGetLastError();
}

}  // namespace rppa

// Validation follows rppt_tensor_audio_augmentations.cpp:539-575.
RPPA_EXPORT RppStatus rppt_resample_gpu(RppPtr_t srcPtr, RpptDescPtr srcDescPtr, RppPtr_t dstPtr,
                                        RpptDescPtr dstDescPtr, Rpp32f *inRateTensor, Rpp32f *outRateTensor,
                                        Rpp32s *srcDimsTensor, RpptResamplingWindow &window, rppHandle_t rppHandle)
{
    if (!rppHandle || !srcDescPtr || !dstDescPtr) return RPP_ERROR_INVALID_ARGUMENTS;
    const size_t dims = srcDescPtr->numDims - 1;
    if (dims != 1 && dims != 2) return RPP_ERROR_INVALID_SRC_DIMS;
    if (srcDescPtr->dataType != F32) return RPP_ERROR_NOT_IMPLEMENTED;
    if (!srcPtr || !dstPtr || !inRateTensor || !outRateTensor || !srcDimsTensor || !window.lookupPinned)
        return RPP_ERROR_INVALID_ARGUMENTS;
    if (window.lookupSize < 2 || window.lookupSize > 16384 || window.lobes < 0) return RPP_ERROR_INVALID_ARGUMENTS;
    const unsigned B = srcDescPtr->n;
    if (B == 0) return RPP_SUCCESS;
    RPPA_HIP(rppa::resample_launch<false>(rppHandle->stream, static_cast<const float *>(srcPtr), srcDescPtr->strides.nStride,
                                          static_cast<float *>(dstPtr), dstDescPtr->strides.nStride, B, inRateTensor,
                                          outRateTensor, srcDimsTensor, window, 0, 0.0f, 0.0f));
    return RPP_SUCCESS;
}

// Down-mix (rppt_down_mixing_gpu's arithmetic) and resample (rppt_resample_gpu's) in one launch:
// src interleaved [n][samples * channels], srcDimsTensor[2b] = samples, [2b+1] = channels; dst
// mono [n][nStride].  Bit-identical to the two calls in sequence; the down-mixed signal never
// goes to memory.
RPPA_EXPORT RppStatus rppt_down_mix_resample_gpu(RppPtr_t srcPtr, RpptDescPtr srcDescPtr, RppPtr_t dstPtr,
                                                 RpptDescPtr dstDescPtr, Rpp32f *inRateTensor, Rpp32f *outRateTensor,
                                                 Rpp32s *srcDimsTensor, bool normalizeWeights,
                                                 RpptResamplingWindow &window, rppHandle_t rppHandle)
{
    if (!rppHandle || !srcDescPtr || !dstDescPtr) return RPP_ERROR_INVALID_ARGUMENTS;
    const size_t dims = srcDescPtr->numDims - 1;
    if (dims != 1 && dims != 2) return RPP_ERROR_INVALID_SRC_DIMS;
    if (srcDescPtr->dataType != F32 || dstDescPtr->dataType != F32) return RPP_ERROR_NOT_IMPLEMENTED;
    if (!srcPtr || !dstPtr || !inRateTensor || !outRateTensor || !srcDimsTensor || !window.lookupPinned)
        return RPP_ERROR_INVALID_ARGUMENTS;
    if (window.lookupSize < 2 || window.lookupSize > 16384 || window.lobes < 0) return RPP_ERROR_INVALID_ARGUMENTS;
    const unsigned B = srcDescPtr->n;
    if (B == 0) return RPP_SUCCESS;
    RPPA_HIP(rppa::resample_launch<true>(rppHandle->stream, static_cast<const float *>(srcPtr), srcDescPtr->strides.nStride,
                                          static_cast<float *>(dstPtr), dstDescPtr->strides.nStride, B, inRateTensor,
                                          outRateTensor, srcDimsTensor, window, normalizeWeights ? 1 : 0, 0.0f, 0.0f));
    return RPP_SUCCESS;
}
