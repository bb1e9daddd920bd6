// spectrogram.hip -- rppt_spectrogram_gpu (api/rppt_tensor_audio_augmentations.h:232), FP32.
//
// Semantics of cpu/kernel/spectrogram.cpp:71-251: F = L/H + 1 centered frames (else (L-W)/H + 1),
// frame f starts at f*H - (center ? W/2 : 0), out-of-range samples are mirrored without
// repeating the edge (reflect) or zero, the frame is multiplied by the window, and bin
// k in [0, N/2] gets |X_k|^2 when power == 2 and |X_k| for any other value -- the rule of the
// GPU entry point this replaces (hip/kernel/spectrogram.cpp:231-232; the HOST kernel instead
// takes |X_k| only for power == 1, cpu/kernel/spectrogram.cpp:217-242).  NFT writes
// dst[k*hStride + f], NTF writes dst[f*hStride + k]; only frames < F are written.
//
// nfft a power of two from 64 to 2048 runs by FFT (fft_real.hpp, spectrogram_fft_kernel below).  Every
// other nfft runs as a dense FP32 contraction  C[f][c] = sum_t x[f*H - off + t] * basis[t][c]  against
// the window-folded basis of tables.hip (the window multiply happens once, in FP64, when the
// basis is built).  The framing is implicit: the A tile is gathered straight from the signal
// with the reflect mapping, so no frame matrix ever goes to HBM (the reference writes
// B*maxFrames*nfft floats of frames and reads them back, hip/kernel/spectrogram.cpp:100-143).
//
// Tiling of the dense contraction (one block = 32 frames of one clip, 256 threads = 4 waves):
//   per K step of 16 samples the block stages A[16][32] and basis[16][512] in LDS; each thread
//   owns 4 frames x 8 re/im column pairs (pairs cg, cg + 32, ... so consecutive lanes read
//   consecutive LDS words) of the 32 x 512 output tile in registers;
//   power is formed in registers, staged in LDS and stored coalesced along frames (NFT) or
//   bins (NTF).  Columns beyond 512 (nfft > 512) are processed in further 512-column passes.
#include "common.hpp"
#include "fft_real.hpp"
#include "tile_plan.hpp"

#include <algorithm>

namespace rppa {
namespace {

constexpr int kFT = 32;      // frames per block
constexpr int kKC = 16;      // K step
constexpr int kCC = 512;     // columns per pass
constexpr int kThreads = 256;
constexpr int kStage = (kKC * kCC > kFT * (kCC / 2 + 1)) ? kKC * kCC : kFT * (kCC / 2 + 1);

struct SpecArgs {
    const float *src;
    uint32_t srcStride;
    const int *lengths;
    float *dst;
    uint32_t dstNStride, hStride;
    int nft;
    int center, reflect;
    int N, W, H, power, cols;
    const float *basis;  // [W][cols]
    const double *rfft;  // the FFT kernel's tables
    int maxFrames;       // frames a clip's output holds
    unsigned tilesX;     // its tiles per clip at most
    int B, plan;         // clips; whether the blocks plan their tiles
};

__device__ inline float sample_at(const float *x, int L, int i, int reflect)
{
    if (i >= 0 && i < L) return x[i];
    if (L <= 0) return 0.0f;
    if (reflect) return x[idx_reflect(i, L)];
    return 0.0f;
}

__global__ void __launch_bounds__(kThreads)
spectrogram_fp32_kernel(SpecArgs a)
{
    __shared__ float sA[kKC][kFT];          // A chunk, [t][f]
    __shared__ float sB[kStage];            // basis chunk [t][c]; reused as the power stage
    const int b = blockIdx.y;
    const int L = min(a.lengths[b], static_cast<int>(a.srcStride));  // never read past the clip's row
    const int F = num_windows(L, a.W, a.H, a.center != 0);
    const int f0 = blockIdx.x * kFT;
    if (f0 >= F) return;
    const float *x = a.src + static_cast<size_t>(b) * a.srcStride;
    const int off = a.center ? a.W / 2 : 0;
    const int tid = threadIdx.x;
    const int cg = tid & 31;        // column pairs cg, cg + 32, ..., cg + 224 of a pass
    const int fg = tid >> 5;        // frame group: 4 frames
    const int K = a.N / 2 + 1;
    const int nPasses = (a.cols + kCC - 1) / kCC;
    float *stage = sB;              // [kFT][kCC/2 + 1] power stage after the K loop

    for (int pass = 0; pass < nPasses; pass++) {
        const int cBase = pass * kCC;
        float acc[4][16];
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 16; j++) acc[i][j] = 0.0f;

        for (int t0 = 0; t0 < a.W; t0 += kKC) {
            // stage A: 16 x 32 = 512 values, 2 per thread
            for (int e = tid; e < kKC * kFT; e += kThreads) {
                int tt = e / kFT, ff = e % kFT;
                int t = t0 + tt, f = f0 + ff;
                float v = 0.0f;
                if (t < a.W && f < F) v = sample_at(x, L, f * a.H - off + t, a.reflect);
                sA[tt][ff] = v;
            }
            // stage basis rows t0..t0+15, columns cBase..cBase+511
            for (int e = tid; e < kKC * kCC; e += kThreads) {
                int tt = e / kCC, cc = e % kCC;
                int t = t0 + tt, c = cBase + cc;
                sB[e] = (t < a.W && c < a.cols) ? a.basis[static_cast<size_t>(t) * a.cols + c] : 0.0f;
            }
            __syncthreads();
#pragma unroll 4
            for (int kk = 0; kk < kKC; kk++) {
                float av[4];
#pragma unroll
                for (int i = 0; i < 4; i++) av[i] = sA[kk][fg * 4 + i];
                float bv[16];
#pragma unroll
                for (int j = 0; j < 8; j++) {   // column pair cg + 32 j: consecutive lanes, consecutive pairs
                    const float2 b2 = *reinterpret_cast<const float2 *>(&sB[kk * kCC + 2 * (cg + 32 * j)]);
                    bv[2 * j] = b2.x;
                    bv[2 * j + 1] = b2.y;
                }
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < 16; j++) acc[i][j] = fmaf(av[i], bv[j], acc[i][j]);
            }
            __syncthreads();
        }

        // power into the stage: stage[f][p] for pair p of this pass (pair 0 of pass 0 = DC/Nyquist)
        const int pairsInPass = kCC / 2;
#pragma unroll
        for (int i = 0; i < 4; i++) {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                float re = acc[i][2 * j], im = acc[i][2 * j + 1];
                int p = cg + 32 * j;
                float v;
                float extra = -1.0f;
                if (pass == 0 && p == 0) {
                    v = re * re;            // DC
                    extra = im * im;        // Nyquist (column 1)
                } else {
                    v = re * re + im * im;
                }
                if (a.power == 1) {
                    v = sqrtf(v);
                    if (extra >= 0.0f) extra = sqrtf(extra);
                }
                stage[(fg * 4 + i) * (pairsInPass + 1) + p] = v;
                if (pass == 0 && p == 0) stage[(fg * 4 + i) * (pairsInPass + 1) + pairsInPass] = extra;
            }
        }
        __syncthreads();
        // store: bins of this pass are pass*256 + p (p >= 1, or p == 0 for pass > 0); pass 0 also
        // owns bin 0 (slot 0) and, for even N, bin N/2 (slot 256)
        const int nf = min(kFT, F - f0);
        const int pStart = pass * pairsInPass;
        for (int e = tid; e < (pairsInPass + 1) * kFT; e += kThreads) {
            int slot, f;
            if (a.nft) { slot = e / kFT; f = e % kFT; } else { f = e / (pairsInPass + 1); slot = e % (pairsInPass + 1); }
            if (f >= nf) continue;
            int k;
            if (slot == pairsInPass) {
                if (pass != 0 || (a.N & 1)) continue;
                k = a.N / 2;
            } else {
                k = pStart + slot;
                if (k >= K) continue;
                if (k == a.N / 2 && !(a.N & 1) && k != 0) continue;  // Nyquist comes from column 1
            }
            float v = stage[f * (pairsInPass + 1) + slot];
            size_t o = static_cast<size_t>(b) * a.dstNStride +
                       (a.nft ? static_cast<size_t>(k) * a.hStride + (f0 + f) : static_cast<size_t>(f0 + f) * a.hStride + k);
            a.dst[o] = v;
        }
        __syncthreads();
    }
}

// Persistent blocks over tiles of one clip.  A tile is the frames the block's waves transform at once,
// straight from the signal (a lane's pairs are 2 R2 samples apart, a group's lanes hold consecutive
// pairs); their power goes to an LDS tile [bin][frame], which takes the turn buffers' place, and from
// there to memory in rows of kFrames frames (NFT) or of bins (NTF).  The row pitch puts the frames and
// lanes of a wave's LDS stores on 64 different banks.
// Bound: vector issue (some 850 vector instructions per four frames of 512, two thirds of them FP64 at about 1.6
// times an FP32 one's issue time) and the latency of the table reads and the two barriers around it.
// Measured against the dense contraction below: 128 ragged clips of 0.5-20 s at nfft 512, hop 160
// 913 -> 73 us; 12 clips of 5-30 s at nfft 2048, hop 512 6,218 -> 114 us; 24 clips of 2-10 s at nfft
// 1024, hop 256 1,582 -> 50 us (an FP32 transform, less exact as fft_real.hpp tells, took 45, 60 and 40 us).
// At nfft 2048 a tile is 143,360 B of LDS, so a CU holds one workgroup, whose eight waves (two per SIMD) move in step
// between the barriers of a tile; the data fill all 256 vector registers and 22 more are spilled.  Smaller sizes spill
// scalar registers only.
template <int N>
struct SpecTile {
    using F = RealFft<N>;
    static constexpr int kWaves = N == 2048 ? 8 : 4;
    static constexpr int kFrames = kWaves * F::kGroups;
    static constexpr int kPitch = kFrames + F::kGroups;
    static constexpr int kThr = kWaves * kWave;
    static constexpr int kPwFloats = (F::M + 1) * kPitch, kTurnFloats = kWaves * F::kTurnFloats;
    static constexpr int kLdsFloats = kPwFloats > kTurnFloats ? kPwFloats : kTurnFloats;
    // waves per SIMD aimed at: what the LDS allows, at most 3 above nfft 128 (the data's registers)
    static constexpr int kOcc = N <= 128 ? 4 : N <= 512 ? 3 : 2;
};

typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));

// The power tile to memory, kSqrt: magnitude.
template <int N, bool kSqrt>
__device__ __forceinline__ void store_tile(const SpecArgs &a, const float *pw, float *out, int f0, int nf)
{
    using F = RealFft<N>;
    using T = SpecTile<N>;
    const int tid = threadIdx.x;
    auto value = [&](int k, int f) {
        const float v = pw[k * T::kPitch + f];
        return kSqrt ? sqrtf(v) : v;
    };
    if (a.nft) {
        // rows k = r + i kRows of the tile: the wave's first row is uniform, so a row's address is a
        // scalar base and the lane's 32-bit offset
        constexpr int kRowsW = kWave / T::kFrames > 0 ? kWave / T::kFrames : 1, kRows = kRowsW * T::kWaves;
        const int lane = tid & 63, f = lane % T::kFrames, rw = lane / T::kFrames;
        const int k0 = __builtin_amdgcn_readfirstlane(tid >> 6) * kRowsW;
        float *o = out + static_cast<size_t>(k0) * a.hStride + f0;
        const unsigned lo = rw * a.hStride + f;
        if (f < nf) {
#pragma unroll 4
            for (int i = 0; i < F::M / kRows; i++) {
                o[lo] = value(k0 + rw + i * kRows, f);
                o += static_cast<size_t>(kRows) * a.hStride;
            }
            if (k0 == 0 && rw == 0) o[lo] = value(F::M, f);
        }
    } else {
        for (int f = 0; f < nf; f++) {
            float *o = out + static_cast<size_t>(f0 + f) * a.hStride;
            for (int k = tid; k <= F::M; k += T::kThr) o[k] = value(k, f);
        }
    }
}

template <int N>
__global__ void __launch_bounds__(SpecTile<N>::kThr, SpecTile<N>::kOcc)
spectrogram_fft_kernel(SpecArgs a)
{
    using F = RealFft<N>;
    using T = SpecTile<N>;
    extern __shared__ __attribute__((aligned(16))) float lds[];
    const int off = a.center ? a.W / 2 : 0;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int l = lane & (F::R1 - 1), g = lane / F::R1;
    double *turn = reinterpret_cast<double *>(lds + wave * F::kTurnFloats) + g * F::kGroupPitch;
    float *pw = lds;
    const int Wr = (a.W + 1) & ~1;
    const int fw = wave * F::kGroups;   // the wave's first frame in a tile
    // frames of clip b, at most what its output holds
    auto frames_of = [&](int L) { return max(min(num_windows(L, a.W, a.H, a.center != 0), a.maxFrames), 0); };
    auto length_of = [&](int b) { return min(a.lengths[b], static_cast<int>(a.srcStride)); };   // stay in the row
    int *start = reinterpret_cast<int *>(lds + T::kLdsFloats);
    unsigned tiles = a.tilesX * a.B;   // without a plan: (clip, tile) pairs, some past their clip's end
    if (a.plan) {
        plan_clips<T::kThr>(start, a.B, start + a.B + 1,
                            [&](int b) { return (frames_of(length_of(b)) + T::kFrames - 1) / T::kFrames; });
        tiles = start[a.B];
    }
    for (unsigned round = 0; round * gridDim.x < tiles; round++) {
        const unsigned tile = plan_tile(round, blockIdx.x, gridDim.x);
        if (tile >= tiles) continue;
        const int b = __builtin_amdgcn_readfirstlane(a.plan ? plan_owner(start, a.B, tile) : tile / a.tilesX);
        const int f0 = __builtin_amdgcn_readfirstlane(tile - (a.plan ? start[b] : b * a.tilesX)) * T::kFrames;
        const int L = length_of(b), nf = min(frames_of(L) - f0, T::kFrames);
        if (nf <= 0) continue;
        const float *x = a.src + static_cast<size_t>(b) * a.srcStride;
        double ar[F::R2], ai[F::R2];
        if (fw < nf) {
            const int fl = min(fw + g, nf - 1);   // frames past the clip's last repeat it
            const int s0 = (f0 + fl) * a.H - off;
            float zr[F::kSub][F::R1], zi[F::kSub][F::R1];
            // first and one past the last sample the wave's frames read
            const int sa = (f0 + fw) * a.H - off, se = (f0 + min(fw + F::kGroups, nf) - 1) * a.H - off + Wr;
            const bool near32 = a.H <= (1 << 24);  // the wave's samples lie within 32-bit offsets of each other
            if (sa >= 0 && se <= L && near32) {    // inside the clip: unconditional 8-byte loads
                const char *xs = reinterpret_cast<const char *>(x + sa);
#pragma unroll
                for (int j = 0; j < F::kSub; j++)
#pragma unroll
                    for (int n1 = 0; n1 < F::R1; n1++) {
                        const int t = 2 * (F::R2 * n1 + F::R1 * j + l);
                        const unsigned o = 4u * static_cast<unsigned>(s0 - sa + (t < Wr ? t : 0));
                        const f32x2u v = *reinterpret_cast<const f32x2u *>(xs + o);
                        zr[j][n1] = v.x;
                        zi[j][n1] = v.y;
                    }
            } else if (sa > -L && se < 2 * L && near32) {   // at most one reflection at either end
                const int lo = max(min(sa, 2 * L - 1 - se), 0);   // the lowest index read
                const char *xs = reinterpret_cast<const char *>(x + lo);
                const int refl = a.reflect ? -1 : 0;
                auto edge = [&](int i) {           // reflected, or clamped to the clip for the zeros below
                    const int m = max(i, -i & refl), c = min(m, L - 1 + ((L - 1 - m) & refl));
                    return *reinterpret_cast<const float *>(xs + 4u * static_cast<unsigned>(c - lo));
                };
#pragma unroll
                for (int j = 0; j < F::kSub; j++)
#pragma unroll
                    for (int n1 = 0; n1 < F::R1; n1++) {
                        const int t = 2 * (F::R2 * n1 + F::R1 * j + l), i = s0 + (t < Wr ? t : 0);
                        zr[j][n1] = edge(i);
                        zi[j][n1] = edge(i + 1);
                    }
                if (!a.reflect) {
#pragma unroll
                    for (int j = 0; j < F::kSub; j++)
#pragma unroll
                        for (int n1 = 0; n1 < F::R1; n1++) {
                            const int i = s0 + 2 * (F::R2 * n1 + F::R1 * j + l);
                            zr[j][n1] = i >= 0 && i < L ? zr[j][n1] : 0.0f;
                            zi[j][n1] = i >= -1 && i < L - 1 ? zi[j][n1] : 0.0f;
                        }
                }
            } else {                               // clips shorter than a window: through the turn buffer
                for (int i = 0; i < 2; i++) {
                    F::wave_sync();
#pragma unroll 1
                    for (int n = l; n < F::M; n += F::R1) turn[n] = sample_at(x, L, s0 + 2 * n + i, a.reflect);
                    F::wave_sync();
#pragma unroll
                    for (int j = 0; j < F::kSub; j++)
#pragma unroll
                        for (int n1 = 0; n1 < F::R1; n1++) {
                            const float v = turn[F::R2 * n1 + F::R1 * j + l];
                            if (i == 0) zr[j][n1] = v;
                            else zi[j][n1] = v;
                        }
                }
            }
            F::mask_window(a.W, l, zr, zi);
            F::transform(F::per_frame(a.rfft), turn, lane, zr, zi, ar, ai);
        }
        __syncthreads();                           // every wave is done with its turn buffer
        if (fw < nf) {
            float *pf = pw + fw + g;
            const unsigned long long bad = F::not_finite(lane, ar, ai);
            F::power(F::per_frame(a.rfft), lane, ar, ai, [&](int k, float v) { pf[k * T::kPitch] = v; });
            if (__builtin_expect(bad != 0, 0)) {
                F::wave_sync();
                int col = fw;   // (opaque, as in infinite_power)
                __asm__ volatile("" : "+s"(col));
                F::infinite_power(
                    a.rfft, a.W, lane, bad,
                    [&](int h, int t) { return sample_at(x, L, (f0 + min(col + h, nf - 1)) * a.H - off + t, a.reflect); },
                    [&](int h, int k, float v) { pw[k * T::kPitch + col + h] = v; });
            }
        }
        __syncthreads();
        float *out = a.dst + static_cast<size_t>(b) * a.dstNStride;
        if (a.power == 1) store_tile<N, true>(a, pw, out, f0, nf);
        else store_tile<N, false>(a, pw, out, f0, nf);
        __syncthreads();                           // the next tile's turn buffers take the power tile's place
    }
}

template <int N>
void launch_fft(rppHandle *h, SpecArgs a, unsigned maxFrames)
{
    using T = SpecTile<N>;
    a.tilesX = ceil_div(maxFrames, T::kFrames);
    // as many blocks as run at once, and no more than there are tiles
    const size_t perCU = std::max(1, T::kOcc * 4 / T::kWaves);
    const size_t pairs = static_cast<size_t>(a.tilesX) * a.B;
    const unsigned grid = plan_grid(perCU * h->numCU, pairs);
    // more pairs than blocks: the tiles that exist are counted and dealt evenly (a ragged batch's pairs
    // dealt as they come left some blocks with twice the average).  Fewer: one pair per block at once.
    a.plan = pairs > grid && a.B <= kPlanClips;
    const size_t bytes = sizeof(float) * T::kLdsFloats + (a.plan ? sizeof(int) * (a.B + 1 + T::kWaves) : 0);
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&spectrogram_fft_kernel<N>),
                              hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
    hipLaunchKernelGGL(spectrogram_fft_kernel<N>, dim3(grid), dim3(T::kThr), bytes, h->stream, a);
}

}  // namespace
}  // namespace rppa

// Validation follows rppt_tensor_audio_augmentations.cpp:579-629 (layout NFT/NTF, src dims 1,
// dst dims 2, F32).  W > nfft is rejected (the reference writes past its FFT buffer there).
RPPA_EXPORT RppStatus rppt_spectrogram_gpu(RppPtr_t srcPtr, RpptDescPtr srcDescPtr, RppPtr_t dstPtr,
                                           RpptDescPtr dstDescPtr, Rpp32s *srcLengthTensor, bool centerWindows,
                                           bool reflectPadding, Rpp32f *windowFunction, Rpp32s nfft, Rpp32s power,
                                           Rpp32s windowLength, Rpp32s windowStep, rppHandle_t rppHandle)
{
    if (!rppHandle || !srcDescPtr || !dstDescPtr) return RPP_ERROR_INVALID_ARGUMENTS;
    if (dstDescPtr->layout != NFT && dstDescPtr->layout != NTF) return RPP_ERROR_INVALID_DST_LAYOUT;
    if (srcDescPtr->numDims - 1 != 1) return RPP_ERROR_INVALID_SRC_DIMS;
    if (dstDescPtr->numDims - 1 != 2) return RPP_ERROR_INVALID_DST_DIMS;
    if (srcDescPtr->dataType != F32 || dstDescPtr->dataType != F32) return RPP_ERROR_NOT_IMPLEMENTED;
    if (!srcPtr || !dstPtr || !srcLengthTensor) return RPP_ERROR_INVALID_ARGUMENTS;
    if (nfft == 0) nfft = windowLength;
    if (windowLength <= 0 || windowStep <= 0 || nfft < 2 || windowLength > nfft) return RPP_ERROR_INVALID_ARGUMENTS;
    const bool nft = dstDescPtr->layout == NFT;
    const int K = nfft / 2 + 1;
    const unsigned maxFrames = nft ? dstDescPtr->w : dstDescPtr->h;
    const unsigned B = srcDescPtr->n;
    if (B == 0 || maxFrames == 0) return RPP_SUCCESS;
    if (nft ? (dstDescPtr->strides.hStride < maxFrames) : (dstDescPtr->strides.hStride < static_cast<unsigned>(K)))
        return RPP_ERROR_INVALID_DST_DIMS;

    const rppa::DftTables *t = rppa::get_dft_tables(rppHandle, nfft, windowLength, windowFunction, -1);
    if (!t) return RPP_ERROR;
    rppa::SpecArgs a;
    a.src = static_cast<const float *>(srcPtr);
    a.srcStride = srcDescPtr->strides.nStride;
    a.lengths = srcLengthTensor;
    a.dst = static_cast<float *>(dstPtr);
    a.dstNStride = dstDescPtr->strides.nStride;
    a.hStride = dstDescPtr->strides.hStride;
    a.nft = nft;
    a.center = centerWindows;
    a.reflect = reflectPadding;
    a.N = nfft;
    a.W = windowLength;
    a.H = windowStep;
    a.power = power == 2 ? 2 : 1;   // the kernel's flag: 1 = magnitude, 2 = squared magnitude
    a.cols = t->cols;
    a.basis = t->basis;
    a.rfft = t->rfft;
    // frames of a clip past the descriptor's are stored up to the next multiple of 32, as far as the row (NFT) or the
    // clip's buffer (NTF) holds them: the dense contraction's rule, which stores whole tiles
    const unsigned room = nft ? a.hStride : a.dstNStride / a.hStride;
    const unsigned fftFrames = std::max(maxFrames, std::min(rppa::ceil_div(maxFrames, rppa::kFT) * rppa::kFT, room));
    a.maxFrames = static_cast<int>(std::min(fftFrames, 0x7fffffffu));
    a.B = static_cast<int>(B);
    switch (rppa::rfft_supported(nfft) ? nfft : 0) {
    case 64: rppa::launch_fft<64>(rppHandle, a, fftFrames); break;
    case 128: rppa::launch_fft<128>(rppHandle, a, fftFrames); break;
    case 256: rppa::launch_fft<256>(rppHandle, a, fftFrames); break;
    case 512: rppa::launch_fft<512>(rppHandle, a, fftFrames); break;
    case 1024: rppa::launch_fft<1024>(rppHandle, a, fftFrames); break;
    case 2048: rppa::launch_fft<2048>(rppHandle, a, fftFrames); break;
    default:
        hipLaunchKernelGGL(rppa::spectrogram_fp32_kernel, dim3(rppa::ceil_div(maxFrames, rppa::kFT), B),
                           dim3(rppa::kThreads), 0, rppHandle->stream, a);
    }
    RPPA_HIP(hipGetLastError());
    return RPP_SUCCESS;
}
