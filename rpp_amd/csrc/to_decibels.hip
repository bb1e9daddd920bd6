// to_decibels.hip -- rppt_to_decibels_gpu (api/rppt_tensor_audio_augmentations.h:122).
//
// out = (multiplier * log10(2)) * log2(max(minRatio, x * (1/ref)))  with
// minRatio = 10^(cutOffDB/multiplier) (0 -> smallest subnormal) and ref = referenceMagnitude, or
// the clip's maximum when referenceMagnitude == 0 (cpu/kernel/to_decibels.cpp:27-99).
// srcDims[b] = {width = columns, height = rows}; width == 1 means 1-D data of `height` samples.
// log2 is evaluated in FP64 and rounded once, the correctly rounded FP32 log2 the HOST path's
// log2f returns, so outputs are bit-identical to RPP HOST.  No host synchronisation (the reference
// synchronises twice, hip/kernel/to_decibels.cpp:283, :295).
//
// Work split: a unit is 256 columns of one row, taken by a wave as four consecutive columns per lane;
// the waves of a clip's blocks stride over its units.  HBM-bound at 8 bytes per value (12 for the
// clip maximum's extra read).  The clip maximum is a partial maximum per block in a buffer of the handle, reduced
// again by every block of the second kernel: one atomic per row and block instead serialised on the
// clips' shared cache line (12 clips of 1,025 rows: 1,396 -> 11 us; the conversion, one value per
// thread in 256-column blocks of one row, 67 -> 17 us on the mel spectra of 128 ragged clips, 80 rows; 21 us of it
// with log2 by a division and a series instead of the table of log2_math.hpp).
#include "common.hpp"
#include "log2_math.hpp"

#include <algorithm>
#include <cfloat>
#include <cmath>

namespace rppa {
namespace {

constexpr int kThreads = 256;

constexpr int kWaves = kThreads / kWave;
constexpr int kUnit = 4 * kWave;     // columns of a unit
constexpr int kMaxChunks = 512;      // blocks per clip

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// The rows and columns of clip b that both buffers hold.
struct DbShape {
    unsigned rows, cols, units, perRow;
    __device__ DbShape(RpptImagePatch d, uint32_t nStride, uint32_t hStride)
    {
        const bool oneD = d.width == 1;
        rows = oneD ? 1 : d.height;
        cols = oneD ? min(d.height, nStride) : min(d.width, hStride);
        perRow = (cols + kUnit - 1) / kUnit;
        units = rows * perRow;
    }
};

__global__ void __launch_bounds__(kThreads)
clip_max_kernel(const float *__restrict__ src, uint32_t nStride, uint32_t hStride, uint32_t maxRows,
                const RpptImagePatch *dims, float *__restrict__ partial)
{
    const int b = blockIdx.y;
    DbShape s(dims[b], nStride, hStride);
    s.units = min(s.rows, maxRows) * s.perRow;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const float *x = src + static_cast<size_t>(b) * nStride;
    float m = -FLT_MAX;
    for (unsigned u = blockIdx.x * kWaves + wave; u < s.units; u += gridDim.x * kWaves) {
        const unsigned row = u / s.perRow, c = (u - row * s.perRow) * kUnit + 4 * lane;
        const float *r = x + static_cast<size_t>(row) * hStride;
        if (c + 4 <= s.cols) {
            const f32x4u v = *reinterpret_cast<const f32x4u *>(r + c);
            m = fmaxf(m, fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w)));
        } else {
            for (unsigned i = c; i < s.cols; i++) m = fmaxf(m, r[i]);
        }
    }
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    __shared__ float red[kWaves];
    if (lane == 0) red[wave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        float r = red[0];
        for (int i = 1; i < kWaves; i++) r = fmaxf(r, red[i]);
        partial[static_cast<size_t>(b) * gridDim.x + blockIdx.x] = r;
    }
}

__device__ inline float db_value(float x, float inv, float minRatio, float mult, const Log2Lds &table)
{
    float v = x * inv;
    float m = (minRatio < v) ? v : minRatio;   // std::max(minRatio, v)
    return mult * log2_rn(m, table);
}

__global__ void __launch_bounds__(kThreads)
to_db_kernel(const float *__restrict__ src, uint32_t srcNStride, uint32_t srcHStride, float *__restrict__ dst,
             uint32_t dstNStride, uint32_t dstHStride, uint32_t maxRows, const RpptImagePatch *dims, float minRatio,
             float mult, float refMag, const float *__restrict__ partial)
{
    __shared__ Log2Lds table;
    table.fill();
    const int b = blockIdx.y;
    DbShape s(dims[b], min(srcNStride, dstNStride), min(srcHStride, dstHStride));
    s.units = min(s.rows, maxRows) * s.perRow;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    unsigned u = blockIdx.x * kWaves + wave;
    if (u >= s.units) return;
    float ref = refMag;
    if (partial) {   // the clip's maximum, of its blocks' partial maxima
        const float *p = partial + static_cast<size_t>(b) * gridDim.x;
        ref = -FLT_MAX;
        for (unsigned i = lane; i < gridDim.x; i += kWave) ref = fmaxf(ref, p[i]);
        for (int o = 32; o > 0; o >>= 1) ref = fmaxf(ref, __shfl_xor(ref, o));
    }
    const float inv = (ref != 0.0f) ? (1.f / ref) : 1.0f;
    const float *x = src + static_cast<size_t>(b) * srcNStride;
    float *y = dst + static_cast<size_t>(b) * dstNStride;
    for (; u < s.units; u += gridDim.x * kWaves) {
        const unsigned row = u / s.perRow, c = (u - row * s.perRow) * kUnit + 4 * lane;
        const float *r = x + static_cast<size_t>(row) * srcHStride;
        float *o = y + static_cast<size_t>(row) * dstHStride;
        if (c + 4 <= s.cols) {
            f32x4u v = *reinterpret_cast<const f32x4u *>(r + c);
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = db_value(v[i], inv, minRatio, mult, table);
            *reinterpret_cast<f32x4u *>(o + c) = v;
        } else {
            for (unsigned i = c; i < s.cols; i++) o[i] = db_value(r[i], inv, minRatio, mult, table);
        }
    }
}

}  // namespace
}  // namespace rppa

// Validation follows rppt_tensor_audio_augmentations.cpp:373-412.
RPPA_EXPORT RppStatus rppt_to_decibels_gpu(RppPtr_t srcPtr, RpptDescPtr srcDescPtr, RppPtr_t dstPtr,
                                           RpptDescPtr dstDescPtr, RpptImagePatchPtr srcDims, Rpp32f cutOffDB,
                                           Rpp32f multiplier, Rpp32f referenceMagnitude, rppHandle_t rppHandle)
{
    if (!rppHandle || !srcDescPtr || !dstDescPtr) return RPP_ERROR_INVALID_ARGUMENTS;
    const size_t dims = srcDescPtr->numDims - 1;
    if (dims != 1 && dims != 2) return RPP_ERROR_INVALID_SRC_DIMS;
    if (!multiplier) return RPP_ERROR_ZERO_DIVISION;
    if (srcDescPtr->dataType != F32) return RPP_ERROR_NOT_IMPLEMENTED;
    if (!srcPtr || !dstPtr || !srcDims) return RPP_ERROR_INVALID_ARGUMENTS;
    const unsigned B = srcDescPtr->n;
    if (B == 0) return RPP_SUCCESS;

    // host-side constants exactly as cpu/kernel/to_decibels.cpp:38-43 computes them
    float minRatio = static_cast<float>(std::pow(10.0, static_cast<double>(cutOffDB / multiplier)));
    if (minRatio == 0.0f) minRatio = std::nextafter(0.0f, 1.0f);
    const float log10Factor = 0.3010299956639812f;
    const float mult = multiplier * log10Factor;

    // grid: x over a clip's units (as many blocks as its largest shape fills, fewer per clip in large
    // batches, at least eight blocks per CU in all), y over clips
    const bool oneD = dims == 1;
    const unsigned cols = oneD ? srcDescPtr->strides.nStride : srcDescPtr->strides.hStride;
    const unsigned rows = oneD ? 1 : std::max(1u, srcDescPtr->h);
    const size_t units = static_cast<size_t>(rppa::ceil_div(cols, rppa::kUnit)) * rows;
    const unsigned most = std::max(1u, std::min<unsigned>(rppa::kMaxChunks, 16u * rppHandle->numCU / B));
    const unsigned gx = std::max(1u, std::min(most, rppa::ceil_div(units, rppa::kWaves)));
    const dim3 grid(gx, B);
    float *partial = nullptr;
    if (referenceMagnitude == 0.0f) {
        partial = static_cast<float *>(rppa::db_workspace(rppHandle, sizeof(float) * gx * B));
        if (!partial) return RPP_ERROR_NOT_ENOUGH_MEMORY;
        hipLaunchKernelGGL(rppa::clip_max_kernel, grid, dim3(rppa::kThreads), 0, rppHandle->stream,
                           static_cast<const float *>(srcPtr), srcDescPtr->strides.nStride, srcDescPtr->strides.hStride,
                           rows, srcDims, partial);
    }
    hipLaunchKernelGGL(rppa::to_db_kernel, grid, dim3(rppa::kThreads), 0, rppHandle->stream,
                       static_cast<const float *>(srcPtr), srcDescPtr->strides.nStride, srcDescPtr->strides.hStride,
                       static_cast<float *>(dstPtr), dstDescPtr->strides.nStride, dstDescPtr->strides.hStride, rows,
                       srcDims, minRatio, mult, referenceMagnitude, partial);
    RPPA_HIP(hipGetLastError());
    return RPP_SUCCESS;
}
