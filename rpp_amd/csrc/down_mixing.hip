// down_mixing.hip -- rppt_down_mixing_gpu (api/rppt_tensor_audio_augmentations.h:188).
//
// mono[t] = sum_c x[t*C + c] * w_c with w_c = 1/C (renormalised to unit sum when
// normalizeWeights), srcDimsTensor[2b] = samples, [2b+1] = channels, interleaved input
// (cpu/kernel/down_mixing.cpp:28-122).  The summation order is the HOST path's: channels in
// groups of 4 (C < 8) or 8 (C >= 8) accumulate lane-wise, the lanes are added as its horizontal
// add does ((l0+l1)+(l2+l3); eight lanes ((l0+l4)+(l2+l6))+((l1+l5)+(l3+l7))), then the leftover
// channels one by one -- so the output is bit-identical to RPP HOST.  (RPP's HIP kernel ignores
// normalizeWeights and sums in a different order, hip/kernel/down_mixing.cpp:28-70.)
// HBM-bound: 4*(C+1) bytes per sample.  One launch serves every channel count (each block reads its
// clip's): stereo takes four outputs per thread from two 16-byte loads and one 16-byte store at any
// 4-byte alignment, other counts one output per thread and step.  32 clips of 3-15 s stereo at 44.1 kHz:
// 19 us; a second launch for the other counts, whose blocks all found stereo and left, cost 18 us more.
#include "common.hpp"
#include "down_mix_math.hpp"

namespace rppa {
namespace {

constexpr int kThreads = 256;

constexpr int kPerThread = 4;

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

__global__ void __launch_bounds__(kThreads)
down_mix_kernel(const float *__restrict__ src, uint32_t srcStride, float *__restrict__ dst, uint32_t dstStride,
                const int *__restrict__ dims, int normalize)
{
    const int b = blockIdx.y;
    const int C = dims[2 * b + 1];
    if (C <= 0) return;
    const long long S = min(static_cast<long long>(dims[2 * b]),
                            min(static_cast<long long>(srcStride) / C, static_cast<long long>(dstStride)));
    const long long base = static_cast<long long>(blockIdx.x) * kThreads * kPerThread;
    if (base >= S) return;
    const float *src0 = src + static_cast<size_t>(b) * srcStride;
    float *y = dst + static_cast<size_t>(b) * dstStride;
    const float w = down_mix_weight(C, normalize);
    if (C == 2) {
        const long long t = base + threadIdx.x * kPerThread;
        if (t >= S) return;
        const float *x = src0 + 2 * t;
        if (t + 4 <= S) {
            const f32x4u p = *reinterpret_cast<const f32x4u *>(x), q = *reinterpret_cast<const f32x4u *>(x + 4);
            const float l0[2] = {p.x, p.y}, l1[2] = {p.z, p.w}, l2[2] = {q.x, q.y}, l3[2] = {q.z, q.w};
            *reinterpret_cast<f32x4u *>(y + t) = f32x4u{down_mix_sample(l0, 2, w), down_mix_sample(l1, 2, w),
                                                        down_mix_sample(l2, 2, w), down_mix_sample(l3, 2, w)};
        } else {
            for (long long u = 0; u < S - t; u++) y[t + u] = down_mix_sample(x + 2 * u, 2, w);
        }
        return;
    }
    for (int i = 0; i < kPerThread; i++) {
        const long long t = base + i * kThreads + threadIdx.x;
        if (t < S) y[t] = down_mix_sample(src0 + t * C, C, w);
    }
}

}  // namespace
}  // namespace rppa

// Validation follows rppt_tensor_audio_augmentations.cpp:416-448.
RPPA_EXPORT RppStatus rppt_down_mixing_gpu(RppPtr_t srcPtr, RpptDescPtr srcDescPtr, RppPtr_t dstPtr,
                                           RpptDescPtr dstDescPtr, Rpp32s *srcDimsTensor, bool normalizeWeights,
                                           rppHandle_t rppHandle)
{
    if (!rppHandle || !srcDescPtr || !dstDescPtr) return RPP_ERROR_INVALID_ARGUMENTS;
    const size_t dims = srcDescPtr->numDims - 1;
    if (dims != 1 && dims != 2) return RPP_ERROR_INVALID_SRC_DIMS;
    if (srcDescPtr->dataType != F32 || dstDescPtr->dataType != F32) return RPP_ERROR_NOT_IMPLEMENTED;
    if (!srcPtr || !dstPtr || !srcDimsTensor) return RPP_ERROR_INVALID_ARGUMENTS;
    const unsigned B = srcDescPtr->n;
    if (B == 0) return RPP_SUCCESS;
    dim3 grid(rppa::ceil_div(dstDescPtr->strides.nStride, rppa::kThreads * rppa::kPerThread), B);
    hipLaunchKernelGGL(rppa::down_mix_kernel, grid, dim3(rppa::kThreads), 0, rppHandle->stream,
                       static_cast<const float *>(srcPtr), srcDescPtr->strides.nStride, static_cast<float *>(dstPtr),
                       dstDescPtr->strides.nStride, srcDimsTensor, normalizeWeights ? 1 : 0);
    RPPA_HIP(hipGetLastError());
    return RPP_SUCCESS;
}
