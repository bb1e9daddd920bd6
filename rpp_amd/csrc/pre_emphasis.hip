// pre_emphasis.hip -- rppt_pre_emphasis_filter_gpu (api/rppt_tensor_audio_augmentations.h:156).
//
// y[0] = x[0] - c*border (border: CLAMP x[0], REFLECT x[1], ZERO 0), y[t] = x[t] - c*x[t-1]
// for t < srcLengthTensor[b] (cpu/kernel/pre_emphasis_filter.cpp:27-75).  The product is
// rounded before the subtraction (no FMA), matching the reference's -mno-fma build, so the
// output is bit-identical to RPP HOST.  HBM-bound, 8 bytes per sample: a lane takes four consecutive
// samples as one 16-byte load and store (any 4-byte alignment), its predecessor comes from the lane
// before it, and kSteps of them are in flight per thread.  128 ragged clips of 0.5-20 s (87 MB): 27 ->
// 16 us (four 4-byte loads and stores 16 bytes apart between lanes before).
#include "common.hpp"

namespace rppa {
namespace {

constexpr int kThreads = 256;
constexpr int kSteps = 4;                              // 16-byte groups per thread
constexpr int kPerBlock = kThreads * 4 * kSteps;       // samples per block

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

__global__ void __launch_bounds__(kThreads)
pre_emphasis_kernel(const float *__restrict__ src, uint32_t srcStride, float *__restrict__ dst, uint32_t dstStride,
                    const int *__restrict__ lengths, const float *__restrict__ coeffs, int border)
{
    const int b = blockIdx.y;
    // a length beyond either stride would run into the next clip; clamp it to the buffer
    const int L = min(lengths[b], static_cast<int>(min(srcStride, dstStride)));
    const size_t base = static_cast<size_t>(blockIdx.x) * kPerBlock;
    if (base >= static_cast<size_t>(max(L, 0))) return;
    const float *x = src + static_cast<size_t>(b) * srcStride + base;
    float *y = dst + static_cast<size_t>(b) * dstStride + base;
    const float c = coeffs[b];
    const unsigned n = min(static_cast<unsigned>(L - base), static_cast<unsigned>(kPerBlock));   // samples of this block
    const int lane = threadIdx.x & 63;
    f32x4u v[kSteps];
    float prev[kSteps];
#pragma unroll
    for (int i = 0; i < kSteps; i++) {
        const unsigned t = (i * kThreads + threadIdx.x) * 4;
        v[i] = f32x4u{0.0f, 0.0f, 0.0f, 0.0f};
        prev[i] = 0.0f;
        if (t + 4 <= n) {
            v[i] = *reinterpret_cast<const f32x4u *>(x + t);
        } else {
            for (unsigned u = t; u < n; u++) v[i][u - t] = x[u];
        }
        if (lane == 0 && t < n && base + t > 0) prev[i] = x[static_cast<ptrdiff_t>(t) - 1];
        if (base + t == 0) prev[i] = border == CLAMP ? v[i][0] : (border == REFLECT && srcStride > 1 ? x[1] : 0.0f);
    }
#pragma unroll
    for (int i = 0; i < kSteps; i++) {
        const unsigned t = (i * kThreads + threadIdx.x) * 4;
        const float before = __shfl_up(v[i][3], 1);
        const float p0 = c * (lane == 0 ? prev[i] : before), p1 = c * v[i][0], p2 = c * v[i][1], p3 = c * v[i][2];
        const f32x4u o = {v[i][0] - p0, v[i][1] - p1, v[i][2] - p2, v[i][3] - p3};
        if (t + 4 <= n) {
            *reinterpret_cast<f32x4u *>(y + t) = o;
        } else {
            for (unsigned u = t; u < n; u++) y[u] = o[u - t];
        }
    }
}

}  // namespace
}  // namespace rppa

// Validation follows rppt_tensor_audio_augmentations.cpp:452-484.
RPPA_EXPORT RppStatus rppt_pre_emphasis_filter_gpu(RppPtr_t srcPtr, RpptDescPtr srcDescPtr, RppPtr_t dstPtr,
                                                   RpptDescPtr dstDescPtr, Rpp32s *srcLengthTensor,
                                                   Rpp32f *coeffTensor, RpptAudioBorderType borderType,
                                                   rppHandle_t rppHandle)
{
    if (!rppHandle || !srcDescPtr || !dstDescPtr) return RPP_ERROR_INVALID_ARGUMENTS;
    if (srcDescPtr->numDims != 2) return RPP_ERROR_INVALID_SRC_DIMS;
    if (srcDescPtr->dataType != F32 || dstDescPtr->dataType != F32) return RPP_ERROR_NOT_IMPLEMENTED;
    if (!srcPtr || !dstPtr || !srcLengthTensor || !coeffTensor) return RPP_ERROR_INVALID_ARGUMENTS;
    const unsigned B = srcDescPtr->n;
    if (B == 0) return RPP_SUCCESS;
    const uint32_t maxLen = srcDescPtr->strides.nStride;
    dim3 grid(rppa::ceil_div(maxLen, rppa::kPerBlock), B);
    hipLaunchKernelGGL(rppa::pre_emphasis_kernel, grid, dim3(rppa::kThreads), 0, rppHandle->stream,
                       static_cast<const float *>(srcPtr), srcDescPtr->strides.nStride, static_cast<float *>(dstPtr),
                       dstDescPtr->strides.nStride, srcLengthTensor, coeffTensor, static_cast<int>(borderType));
    RPPA_HIP(hipGetLastError());
    return RPP_SUCCESS;
}
