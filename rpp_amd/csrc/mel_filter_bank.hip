// mel_filter_bank.hip -- rppt_mel_filter_bank_gpu (api/rppt_tensor_audio_augmentations.h:274), FP32.
//
// out[m][f] = sum_k W[m][k] * S[k][f] over the triangular filters of
// cpu/kernel/mel_filter_bank.cpp:27-198.  The tables come from tables.hip (built on the GPU with
// the reference's algorithm).  Each output adds the rounded products (no FMA) of its filter's bins in
// ascending order from 0 -- the reference's order of operations, so given the same spectrogram and
// tables the result is bit-identical to RPP HOST.
//
// Every bin feeds at most two filters: the one it falls on (interval - 1) and the one it rises on
// (interval).  A lane owns one frame and walks the bins once with two running sums, so a spectrum
// value is read once (a thread per filter and frame read it twice, in blocks of one filter).  The
// filters are split into groups of about equal bin counts, one wave each, for enough waves in flight;
// a group also reads its last filter's falling bins, the next group's first interval.  Weights and
// interval ends are wave-uniform (scalar loads), kMelAhead rows are in flight per lane, and
// consecutive lanes take consecutive frames, so reads and writes are coalesced.  HBM-bound: 128
// ragged clips of 0.5-20 s, 257 bins, 80 filters (92 MB): 97 -> 28 us.
#include "common.hpp"

#include <algorithm>

namespace rppa {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;

template <typename T>
__device__ __forceinline__ T ld_const(const T *p, int i)   // wave-uniform index: a scalar load
{
    typedef const __attribute__((address_space(4))) T *ConstPtr;
    return ((ConstPtr)p)[i];
}

__global__ void __launch_bounds__(kThreads)
mel_bands_kernel(const float *__restrict__ src, uint32_t srcNStride, uint32_t srcHStride,
                 float *__restrict__ dst, uint32_t dstNStride, uint32_t dstHStride, const int *__restrict__ srcDims,
                 const float *__restrict__ pairs, const int *__restrict__ ivStart, int M, int groups)
{
    const int b = blockIdx.z;
    const int F = min(srcDims[2 * b + 1], static_cast<int>(min(srcHStride, dstHStride)));
    const int f0 = blockIdx.x * kWave;
    if (f0 >= F) return;
    const int lane = threadIdx.x & 63;
    const int g = blockIdx.y * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // the group's filters [mA, mB): those whose rising bins start within its share of the bins
    const int k0 = ld_const(ivStart, 0), nk = ld_const(ivStart, M + 1) - k0;
    const int cutA = k0 + static_cast<int>(static_cast<long long>(nk) * g / groups);
    const int cutB = k0 + static_cast<int>(static_cast<long long>(nk) * (g + 1) / groups);
    int mA = 0, mB = 0;
    for (int m = lane; m - lane < M; m += kWave) {
        const int s = ivStart[min(m, M - 1)];
        mA += __popcll(__ballot(m < M && s < cutA));
        mB += __popcll(__ballot(m < M && s < cutB));
    }
    if (g == 0) mA = 0;
    if (g == groups - 1) mB = M;
    if (mA >= mB) return;
    const int f = f0 + lane, fc = min(f, F - 1);
    const float *s = src + static_cast<size_t>(b) * srcNStride + fc;
    float *o = dst + static_cast<size_t>(b) * dstNStride + f;
    const int kA = ld_const(ivStart, mA), kB = ld_const(ivStart, mB + 1);
    int iv = mA, end = ld_const(ivStart, iv + 1), next = ld_const(ivStart, min(iv + 2, M + 1));
    float down = 0.0f, up = 0.0f;   // running sums of filters iv - 1 and iv
    auto close = [&]() {            // interval iv is done: filter iv - 1 is complete
        if (iv > mA && f < F) o[static_cast<size_t>(iv - 1) * dstHStride] = down;
        down = up;
        up = 0.0f;
        iv++;
        end = next;
        next = ld_const(ivStart, min(iv + 2, M + 1));
    };
    float v[kMelAhead], w[2 * kMelAhead];
#pragma unroll
    for (int i = 0; i < kMelAhead; i++) v[i] = s[static_cast<size_t>(min(kA + i, kB - 1 > 0 ? kB - 1 : 0)) * srcHStride];
#pragma unroll
    for (int i = 0; i < 2 * kMelAhead; i++) w[i] = ld_const(pairs, 2 * kA + i);
    for (int k = kA; k < kB; k += kMelAhead) {
        float c[kMelAhead], wc[2 * kMelAhead];
#pragma unroll
        for (int i = 0; i < kMelAhead; i++) c[i] = v[i];
#pragma unroll
        for (int i = 0; i < 2 * kMelAhead; i++) {
            wc[i] = w[i];
            w[i] = ld_const(pairs, 2 * (k + kMelAhead) + i);
        }
#pragma unroll
        for (int i = 0; i < kMelAhead; i++) v[i] = s[static_cast<size_t>(min(k + kMelAhead + i, kB - 1)) * srcHStride];
#pragma unroll
        for (int i = 0; i < kMelAhead; i++) {
            if (k + i < kB) {
                while (k + i >= end) close();
                const float p = c[i] * wc[2 * i], q = c[i] * wc[2 * i + 1];
                down = down + p;
                up = up + q;
            }
        }
    }
    while (iv <= mB) close();
}

}  // namespace
}  // namespace rppa

// Validation follows rppt_tensor_audio_augmentations.cpp:488-535.  numBins is srcDesc->h, as the
// reference HIP path takes it (hip/kernel/mel_filter_bank.cpp:163-167).
RPPA_EXPORT RppStatus rppt_mel_filter_bank_gpu(RppPtr_t srcPtr, RpptDescPtr srcDescPtr, RppPtr_t dstPtr,
                                               RpptDescPtr dstDescPtr, Rpp32s *srcDims, Rpp32f maxFreq, Rpp32f minFreq,
                                               RpptMelScaleFormula melFormula, Rpp32s numFilter, Rpp32f sampleRate,
                                               bool normalize, rppHandle_t rppHandle)
{
    if (!rppHandle || !srcDescPtr || !dstDescPtr) return RPP_ERROR_INVALID_ARGUMENTS;
    if (srcDescPtr->numDims - 1 != 2) return RPP_ERROR_INVALID_SRC_DIMS;
    if (srcDescPtr->layout != NFT) return RPP_ERROR_INVALID_SRC_LAYOUT;
    if (dstDescPtr->layout != NFT) return RPP_ERROR_INVALID_DST_LAYOUT;
    if (maxFreq < 0 || maxFreq > sampleRate / 2) return RPP_ERROR_INVALID_ARGUMENTS;
    if (minFreq < 0 || minFreq > sampleRate / 2) return RPP_ERROR_INVALID_ARGUMENTS;
    if (srcDescPtr->dataType != F32 || dstDescPtr->dataType != F32) return RPP_ERROR_NOT_IMPLEMENTED;
    if (!srcPtr || !dstPtr || !srcDims || numFilter <= 0 || srcDescPtr->h < 2) return RPP_ERROR_INVALID_ARGUMENTS;
    const unsigned B = srcDescPtr->n;
    const unsigned maxFrames = dstDescPtr->w;
    if (B == 0 || maxFrames == 0) return RPP_SUCCESS;
    const rppa::MelTables *t = rppa::get_mel_tables(rppHandle, static_cast<int>(srcDescPtr->h), sampleRate, maxFreq,
                                                    minFreq, static_cast<int>(melFormula), numFilter, normalize ? 1 : 0);
    if (!t) return RPP_ERROR;
    // 8 filter groups, up to 64 where they would leave the chip short of waves (4,096, four per SIMD).  One clip of 200
    // frames, 80 filters: 5.4 us with 16 groups, 4.6 with 64; 8 clips of 100-300 frames, 256 filters 8.9 and 6.1
    // (frames of a clip past the descriptor's width are formed up to the next multiple of 256, as far as rows hold them)
    const unsigned chunks = rppa::ceil_div(std::max(maxFrames, std::min((maxFrames + 255) / 256 * 256,
                                                                        std::min(srcDescPtr->strides.hStride, dstDescPtr->strides.hStride))),
                                           rppa::kWave);
    int groups = 8;
    while (groups < 64 && static_cast<size_t>(chunks) * B * groups < 4096) groups *= 2;
    dim3 grid(chunks, groups / rppa::kWaves, B);
    hipLaunchKernelGGL(rppa::mel_bands_kernel, grid, dim3(rppa::kThreads), 0, rppHandle->stream,
                       static_cast<const float *>(srcPtr), srcDescPtr->strides.nStride, srcDescPtr->strides.hStride,
                       static_cast<float *>(dstPtr), dstDescPtr->strides.nStride, dstDescPtr->strides.hStride, srcDims,
                       reinterpret_cast<const float *>(t->pairs), t->ivStart, numFilter, groups);
    RPPA_HIP(hipGetLastError());
    return RPP_SUCCESS;
}
