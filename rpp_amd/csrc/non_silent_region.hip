// non_silent_region.hip -- rppt_non_silent_region_detection_gpu
// (api/rppt_tensor_audio_augmentations.h:86).
//
// Semantics of the HOST kernel (src/modules/tensor/cpu/kernel/non_silent_region_detection.cpp:93-191):
// the moving mean square mms[p] = (sum of x[i]^2, p-W < i <= p) / W is a running FP32 sum that
// is restarted every resetInterval outputs (from a fresh sum of the W-1 samples before the
// block); the region runs from the first to the last p with mms[p] >= base * 10^(cutOffDB/10),
// base = max(mms) (referencePower == 0) or referencePower, and its begin is moved W-1 samples
// earlier (clamped at 0) unless it is 0.
//
// The running sum is evaluated in the HOST order (add the square, scale, subtract the square
// leaving the window; products rounded before the add, as the reference's -mno-fma build does),
// so mms is bit-identical to that sequence and the detected indices match it exactly.  The
// reference's HIP kernel uses per-tile prefix sums instead, whose rounding differs from HOST.
//
// Parallelism is the reset blocks: one lane runs one block's recurrence, on squares that other waves of
// its workgroup load and form (batches of 2 GiB and more: one lane does it all).  The recurrence's whole
// state is the running sum, so pass 1 records it every kSeg outputs together with the largest sum
// of those outputs; pass 2, one workgroup per clip, reduces the records to the cut-off (unless the
// reference power fixes it) and resumes the recurrence from the recorded sums over only the two
// kSeg-output spans holding the region's ends.
#include <algorithm>
#include <cmath>

#include "common.hpp"
#include "tile_plan.hpp"

namespace rppa {
namespace {

constexpr int kChunk = 32;          // samples per lane per prefetch step (three steps in flight)
constexpr int kSeg = 192;           // outputs between checkpoints of the running sum
constexpr int kPass1Threads = 64;   // one wave per workgroup spreads the few lanes over CUs
// rows (reset blocks) per pass-1 wave: 32 of the 64 lanes.  Measured on workload 1 (5,378 rows of up
// to 10,240 samples over 512 x 39 lanes, block-major): 64 rows per wave 228.6 us, 32 219.4 us, 16 331 us, 8 515 us; each wave's
// instruction stream is the same for any number of active lanes, and below 32 rows per wave the
// waves outnumber what the compute units run at one wave per SIMD
constexpr int kPass1Rows = 32;
constexpr int kPass2Threads = 128;
// clips up to which the streamed kernel numbers the blocks in LDS: 3,000 clips of 4,000-32,000 samples 148 us with the
// numbering, 198 without; 4,000 clips 240 and 217, 8,000 clips of 1,000-5,000 samples in blocks of 1,000 303 and 149
constexpr int kPlanned = 3072;
static_assert(kSeg % (3 * kChunk) == 0, "checkpoints fall on loop steps");

struct NsrArgs {
    const float *src;
    long long nStride;
    const int *len;
    int W;              // at most nStride + 1: from there on no sample leaves the window, and positions fit 32 bits
    float meanFactor;   // 1 / the caller's window
    int R;              // reset length; <= 0 means the whole clip is one block
    int maxBlocks;
    int segsPerBlock;   // checkpoints per reset block
    int maxSegs;        // checkpoints per clip row
    float cutOff;       // 10^(cutOffDB/10)
    float refPower;     // 0: per-clip maximum
    float *segMax;      // [B][maxSegs] maximum running sum over each checkpoint's outputs
    float *segSum;      // [B][maxSegs] running sum before each checkpoint's first output
    float *blockMax;    // [B][maxBlocks] maximum running sum over each reset block
    int *begin;
    int *length;
    int srcBytes;       // B * nStride * 4 when under 2 GiB, else 0
};

__device__ __forceinline__ int clip_len(const NsrArgs &a, int b)
{
    long long L = a.len[b];
    if (L < 0) L = 0;
    if (L > a.nStride) L = a.nStride;
    return static_cast<int>(L);
}

__device__ __forceinline__ int blocks_of(int L, int R) { return L <= 0 ? 0 : (R <= 0 ? 1 : (L + R - 1) / R); }

// x[i] for i clamped into [0, n): chunk loads may run past either end of a stream; the values
// loaded there are never used.
__device__ __forceinline__ float ld(const float *x, int i, int n) { return x[min(max(i, 0), n - 1)]; }

// Fresh sum of the W-1 squares before output `start`, in order (HOST :129-130).
__device__ __forceinline__ float fresh_sum(const float *x, int n, int start, int W)
{
    float sum = 0.0f;
    const int f0 = max(start - W + 1, 0);
    float b0[kChunk], b1[kChunk], b2[kChunk];
    auto load = [&](float (&v)[kChunk], int i0) {
#pragma unroll
        for (int u = 0; u < kChunk; u++) v[u] = ld(x, i0 + u, n);
    };
    auto add = [&](const float (&v)[kChunk], int i0) {
#pragma unroll
        for (int u = 0; u < kChunk; u++) {
            float q = v[u] * v[u];
            sum = sum + (i0 + u < start ? q : 0.0f);   // adding +0 keeps the sum
        }
    };
    if (f0 < start) {
        load(b0, f0);
        load(b1, f0 + kChunk);
        load(b2, f0 + 2 * kChunk);
        for (int i0 = f0; i0 < start; i0 += 3 * kChunk) {
            add(b0, i0);
            load(b0, i0 + 3 * kChunk);
            add(b1, i0 + kChunk);
            load(b1, i0 + 4 * kChunk);
            add(b2, i0 + 2 * kChunk);
            load(b2, i0 + 5 * kChunk);
        }
    }
    return sum;
}

// Runs the HOST recurrence over outputs [start, end) of one clip of length n from the running
// sum `sum` and calls visit(p, sum_p, p < end) in order, where mms[p] = sum_p * (1/W) rounded;
// mark(off, sum) is called before the outputs start + off of every loop step (off a multiple of
// 3 kChunk) with the sum the recurrence resumes from there.  Branch-free: the recurrence runs on
// to the end of the last chunk (values past `end` are flagged invalid and never used).  The
// recurrence is sequential (its rounding is the HOST's), so the loads run ahead of it: three
// chunks are in flight while one is consumed (the buffers rotate by name in a loop unrolled
// three times, so no values are copied).
template <class Visit, class Mark>
__device__ __forceinline__ void mms_main(const float *x, int n, int start, int end, int W, float sum,
                                         Visit &visit, Mark &mark)
{
    float a0[kChunk], a1[kChunk], a2[kChunk], s0[kChunk], s1[kChunk], s2[kChunk];
    auto load2 = [&](float (&av)[kChunk], float (&sv)[kChunk], int p0) {
#pragma unroll
        for (int i = 0; i < kChunk; i++) {
            av[i] = ld(x, p0 + i, n);
            sv[i] = ld(x, p0 - W + 1 + i, n);
        }
    };
    auto run = [&](const float (&av)[kChunk], const float (&sv)[kChunk], int p0) {
#pragma unroll
        for (int i = 0; i < kChunk; i++) {
            const int p = p0 + i;
            float q = av[i] * av[i];
            sum = sum + q;
            visit(p, sum, p < end);
            float r = sv[i] * sv[i];
            sum = sum - (p - W + 1 >= 0 ? r : 0.0f);   // x - 0 is x: the HOST's skipped subtraction
        }
    };
    load2(a0, s0, start);
    load2(a1, s1, start + kChunk);
    load2(a2, s2, start + 2 * kChunk);
    for (int p0 = start; p0 < end; p0 += 3 * kChunk) {
        mark(p0 - start, sum);
        run(a0, s0, p0);
        load2(a0, s0, p0 + 3 * kChunk);
        run(a1, s1, p0 + kChunk);
        load2(a1, s1, p0 + 4 * kChunk);
        run(a2, s2, p0 + 2 * kChunk);
        load2(a2, s2, p0 + 5 * kChunk);
    }
}

// Loads of samples at .. at + 3 of the whole batch (under 2 GiB) through a buffer resource, at any 4-byte
// alignment.  Reads past a row's end or before its start fall on neighbouring rows, reads past the batch's end
// or before its start give zeros; nothing read there reaches an output.
struct Row4 {
    __amdgpu_buffer_rsrc_t rsrc;
    int samples;   // of the batch

    // The offset is hidden from the optimiser: an immediate offset that it splits off the sum can leave the
    // lane's own offset negative, which the hardware takes as out of range whatever the sum is.
    __device__ __forceinline__ float4 operator()(int at) const
    {
        unsigned o = static_cast<unsigned>(at) * 4u;
        __asm__("" : "+v"(o));
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, o, 0, 0);
        return make_float4(__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3]));
    }
    // sample by sample, each clamped into the batch: for groups that straddle its first or last sample
    __device__ __forceinline__ float4 singles(int at) const
    {
        float v[4];
#pragma unroll
        for (int k = 0; k < 4; k++)
            v[k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                rsrc, static_cast<unsigned>(min(max(at + k, 0), samples - 1)) * 4u, 0, 0));
        return make_float4(v[0], v[1], v[2], v[3]);
    }
};

__device__ __forceinline__ Row4 row4(const NsrArgs &a)
{
    return Row4{__builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.src), 0, a.srcBytes, 0x00020000), a.srcBytes / 4};
}

// The running maximum of the visited sums.
struct RunMax {
    float m = -INFINITY;
    __device__ __forceinline__ void operator()(int, float s, bool valid) { m = fmaxf(m, valid ? s : -INFINITY); }
};

// ---- Pass 1, streamed: producer waves square, one wave adds -------------------------------------
// A workgroup takes eight reset blocks.  Wave 1 loads and squares the samples entering the window, wave 2
// those leaving it, kSeg outputs of every block at a time, into one of two LDS buffers; lane r of wave
// 0 runs block r's recurrence from the other: one addition and one subtraction per sample with the
// running maximum and the 16-byte LDS reads in their latency slots.  The W - 1 squares of the fresh sum
// come the same way first (masked to its range: adding +0 keeps the sum), and trailing samples before
// the clip's start are 0 (x - 0 is x, the HOST's skipped subtraction).  The operations and their order
// are mms_main's.
//
// Bound: the recurrence, two dependent FP32 operations of about 8 cycles each per sample (a wave that is alone on its SIMD
// waits out each operand); a wave that also loads, squares and broadcasts its samples issues 6.4
// instructions per sample, 28 cycles.  Detection on 256 clips of 0.5-20 s, both passes: 146 -> 113 us; 512 clips 147 -> 115 us.
constexpr int kRows = 8;                       // reset blocks per workgroup (16: 120 us, 4: 107 us, but 127 against 115 on 512 clips)
constexpr int kStreamThreads = 3 * kWave;
constexpr int kPitch = kSeg + 4;               // floats per block row of a buffer (64 banks: 4 apart)
constexpr int kVecs = kRows * kSeg / 4 / kWave;   // 16-byte groups per producer lane and chunk
constexpr int kAhead = 2;                      // chunks a producer has in flight
static_assert(kRows * kSeg % (4 * kWave) == 0 && kSeg % 16 == 0, "whole groups per lane");

// Two steps of the recurrence: s += q0 (a0), s -= r0, s += q1 (a1), s -= r1, m = max(m, a0, a1).
__device__ __forceinline__ void mms_pair(float &s, float &m, float q0, float q1, float r0, float r1)
{
    float a0, a1;
    __asm__ volatile("v_add_f32 %[a0], %[s], %[q0]\n\t"
                     "v_sub_f32 %[s], %[a0], %[r0]\n\t"
                     "v_add_f32 %[a1], %[s], %[q1]\n\t"
                     "v_sub_f32 %[s], %[a1], %[r1]\n\t"
                     "v_max3_f32 %[m], %[m], %[a0], %[a1]"
                     : [s] "+v"(s), [m] "+v"(m), [a0] "=&v"(a0), [a1] "=&v"(a1)
                     : [q0] "v"(q0), [q1] "v"(q1), [r0] "v"(r0), [r1] "v"(r1));
}

// planned: the blocks are numbered clip by clip (the prefix of each clip's block count, in LDS), so
// every workgroup but the last holds kRows of them; else (one block per clip, or more clips than
// kPlanned) block j of clip b is number j * B + b and the numbers past a clip's blocks stay idle.
__global__ void __launch_bounds__(kStreamThreads) nsr_blocks_stream_kernel(NsrArgs a, int B, int planned)
{
    __shared__ __attribute__((aligned(16))) float buf[2][2][kRows * kPitch];   // [parity][entering, leaving]
    __shared__ int sStart[kRows], sEnd[kRows], sClip[kRows], sIndex[kRows];
    __shared__ int sRow[kRows];   // first sample of the row in the batch
    extern __shared__ int pre[];   // [B + 1] and the plan's scratch, when planned
    const int tid = static_cast<int>(threadIdx.x), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (planned) plan_clips<kStreamThreads>(pre, B, pre + B + 1, [&](int bb) { return blocks_of(clip_len(a, bb), a.R); });
    if (tid < kRows) {
        const long long row = static_cast<long long>(blockIdx.x) * kRows + tid;
        int b = 0, j = 0, start = 0, end = 0;   // an idle row: no outputs
        bool have = false;
        if (planned) {
            if (row < pre[B]) {
                int lo = 0, hi = B;
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (pre[mid] <= row) lo = mid;
                    else hi = mid;
                }
                b = lo;
                j = static_cast<int>(row) - pre[b];
                have = true;
            }
        } else {
            b = static_cast<int>(row % B);
            j = static_cast<int>(row / B);
            have = j < blocks_of(clip_len(a, b), a.R);
        }
        if (have) {
            const int L = clip_len(a, b);
            const int R = a.R <= 0 ? L : a.R;
            start = j * R;
            end = static_cast<int>(min(static_cast<long long>(L), static_cast<long long>(start) + R));
        }
        sClip[tid] = b;
        sIndex[tid] = j;
        sStart[tid] = start;
        sEnd[tid] = end;
        sRow[tid] = b * static_cast<int>(a.nStride);
    }
    __syncthreads();
    int longest = 0;
    for (int r = 0; r < kRows; r++) longest = max(longest, sEnd[r] - sStart[r]);
    if (longest == 0) return;
    // the fresh sums reach back to the window's or the clip's start: as many chunks as the workgroup's longest
    // needs (by the window alone, a window of 160,000 samples cost 0.5 ms in any batch)
    int fresh = 0;
    for (int r = 0; r < kRows; r++) fresh = max(fresh, min(a.W - 1, sStart[r]));
    fresh = __builtin_amdgcn_readfirstlane(fresh);       // (uniform: scalar loop control)
    longest = __builtin_amdgcn_readfirstlane(longest);
    const int nFresh = (fresh + kSeg - 1) / kSeg;
    const int nChunks = nFresh + (longest + kSeg - 1) / kSeg;

    if (wave > 0) {   // ------------------------------------------------------------ producers
        const bool leaving = wave == 2;
        const Row4 ld4 = row4(a);
        // 16-byte group i of the lane: its position in chunk 0, the first position that counts, its place in the buffer
        int first[kVecs], lo[kVecs], at[kVecs], row[kVecs];   // (row: the position in the batch)
#pragma unroll
        for (int i = 0; i < kVecs; i++) {
            const int f = i * kWave + lane, r = f / (kSeg / 4), col = f % (kSeg / 4) * 4;
            first[i] = sStart[r] - nFresh * kSeg + col - (leaving ? a.W - 1 : 0);
            // entering squares before `start` count from the fresh sum's first on; leaving ones from the clip's start
            lo[i] = leaving ? 0 : max(sStart[r] - a.W + 1, 0);
            at[i] = r * kPitch + col;
            row[i] = sRow[r] + first[i];
        }
        // a group with a sample that counts starts at most three samples before its row and ends at most three
        // past it, so only rows that near to the batch's first or last sample have groups that straddle it
        bool edge = false;
        for (int r = 0; r < kRows; r++)
            edge = edge || sRow[r] < 3 || a.srcBytes / 4 - sRow[r] - static_cast<int>(a.nStride) < 3;
        float4 v[kAhead][kVecs];
        auto load = [&](int u, int c) {
#pragma unroll
            for (int i = 0; i < kVecs; i++) v[u][i] = ld4(row[i] + c * kSeg);
        };
        auto put = [&](int u, int c) {
            if (edge) {
                // straddling groups may lack samples that lie in the batch: the chunk is loaded again, each
                // sample clamped into the batch (the asm has the loads waited for in here: pending past the
                // branch, they would have every chunk's groups waited for as if they were the newest loads)
                bool straddles = false;
#pragma unroll
                for (int i = 0; i < kVecs; i++) {
                    const int p = row[i] + c * kSeg;
                    straddles = straddles || (p < 0 && p > -4) || (p < ld4.samples && p > ld4.samples - 4);
                }
                if (__ballot(straddles) != 0) {
#pragma unroll
                    for (int i = 0; i < kVecs; i++) {
                        v[u][i] = ld4.singles(row[i] + c * kSeg);
                        __asm__ volatile("" : "+v"(v[u][i].x), "+v"(v[u][i].y), "+v"(v[u][i].z), "+v"(v[u][i].w));
                    }
                }
            }
            float *to = buf[c & 1][leaving ? 1 : 0];
#pragma unroll
            for (int i = 0; i < kVecs; i++) {
                const int p = first[i] + c * kSeg;
                const float4 x = v[u][i];
                float4 q = make_float4(x.x * x.x, x.y * x.y, x.z * x.z, x.w * x.w);
                if (p < lo[i]) {
                    q.x = p >= lo[i] ? q.x : 0.0f;
                    q.y = p + 1 >= lo[i] ? q.y : 0.0f;
                    q.z = p + 2 >= lo[i] ? q.z : 0.0f;
                    q.w = p + 3 >= lo[i] ? q.w : 0.0f;
                }
                *reinterpret_cast<float4 *>(to + at[i]) = q;
            }
        };
        // chunk c is put before the barrier that opens the consumer's step c; nothing leaves during the fresh sum
        int c = 0;
        for (const int c0 = leaving ? nFresh / kAhead * kAhead : 0; c < c0; c++) __syncthreads();
#pragma unroll
        for (int u = 0; u < kAhead; u++) load(u, c + u);
        for (; c + kAhead <= nChunks; c += kAhead) {
#pragma unroll
            for (int u = 0; u < kAhead; u++) {
                put(u, c + u);
                load(u, c + u + kAhead);
                __syncthreads();
            }
        }
#pragma unroll
        for (int u = 0; u + 1 < kAhead; u++) {
            if (c + u < nChunks) {
                put(u, c + u);
                __syncthreads();
            }
        }
        return;
    }

    // ---------------------------------------------------------------------------------- consumer
    const int r = lane & (kRows - 1);
    const bool mine = lane < kRows;
    const int start = sStart[r], end = sEnd[r], b = sClip[r], j = sIndex[r];
    float *segMax = a.segMax + static_cast<long long>(b) * a.maxSegs + static_cast<long long>(j) * a.segsPerBlock;
    float *segSum = a.segSum + static_cast<long long>(b) * a.maxSegs + static_cast<long long>(j) * a.segsPerBlock;
    float sum = 0.0f, mb = -INFINITY;
    for (int c = 0; c < nFresh; c++) {
        __syncthreads();
        const float4 *q = reinterpret_cast<const float4 *>(buf[c & 1][0] + r * kPitch);
#pragma unroll 12
        for (int i = 0; i < kSeg / 4; i++) {
            const float4 x = q[i];
            sum = sum + x.x;
            sum = sum + x.y;
            sum = sum + x.z;
            sum = sum + x.w;
        }
    }
    for (int c = nFresh; c < nChunks; c++) {
        __syncthreads();
        const int k = c - nFresh, left = end - start - k * kSeg;   // this block's outputs from here on
        const float4 *q = reinterpret_cast<const float4 *>(buf[c & 1][0] + r * kPitch);
        const float4 *t = reinterpret_cast<const float4 *>(buf[c & 1][1] + r * kPitch);
        const float sum0 = sum;
        float m = -INFINITY;
        if (__ballot(left > 0 && left < kSeg) == 0) {      // (a block that has ended runs on, its sums unused)
            // the squares of a step of 16 samples are read while the step before is added
            float4 qa[4], ta[4], qb[4], tb[4];
            auto read = [&](float4 (&x)[4], float4 (&y)[4], int g) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    x[i] = q[4 * g + i];
                    y[i] = t[4 * g + i];
                }
            };
            auto add = [&](const float4 (&x)[4], const float4 (&y)[4]) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    mms_pair(sum, m, x[i].x, x[i].y, y[i].x, y[i].y);
                    mms_pair(sum, m, x[i].z, x[i].w, y[i].z, y[i].w);
                }
            };
            read(qa, ta, 0);
#pragma unroll 1
            for (int g = 0; g < kSeg / 16; g += 2) {
                read(qb, tb, g + 1);
                add(qa, ta);
                if (g + 2 < kSeg / 16) read(qa, ta, g + 2);
                add(qb, tb);
            }
        } else {
            const float *qs = reinterpret_cast<const float *>(q), *ts = reinterpret_cast<const float *>(t);
            const int steps = min(kSeg, longest - k * kSeg);   // (to the end of the workgroup's longest block)
            for (int i = 0; i < steps; i++) {
                sum = sum + qs[i];
                m = i < left ? fmaxf(m, sum) : m;
                sum = sum - ts[i];
            }
        }
        if (mine && left > 0) {
            segSum[k] = sum0;
            segMax[k] = m;
            mb = fmaxf(mb, m);
        }
    }
    if (mine && end > start) a.blockMax[static_cast<long long>(b) * a.maxBlocks + j] = mb;
}

// Pass 1: one lane per reset block records, every kSeg outputs, the running sum the recurrence
// resumes from and the largest running sum of those outputs, and the block's largest running sum
// (mms = sum * (1/W) rounded is monotone in sum, so the largest mms is the largest sum times 1/W,
// rounded, and a block or span holds an mms >= cut exactly when its largest sum times 1/W does).
__global__ void __launch_bounds__(kPass1Threads) nsr_blocks_kernel(NsrArgs a, int B)
{
    if (threadIdx.x >= kPass1Rows) return;
    const long long lane = static_cast<long long>(blockIdx.x) * kPass1Rows + threadIdx.x;
    if (lane >= static_cast<long long>(B) * a.maxBlocks) return;
    // consecutive lanes take the same block of consecutive clips: the lanes of a wave then read
    // rows a clip stride apart rather than blocks a reset interval apart (a power-of-two stride
    // that sends every lane's load to the same memory channel)
    const int b = static_cast<int>(lane % B);
    const int j = static_cast<int>(lane / B);
    const int L = clip_len(a, b);
    if (j >= blocks_of(L, a.R)) return;
    const int R = a.R <= 0 ? L : a.R;
    const int start = j * R;
    const int end = static_cast<int>(min(static_cast<long long>(L), static_cast<long long>(start) + R));
    const float *x = a.src + b * a.nStride;
    const float sum0 = fresh_sum(x, L, start, a.W);
    float *segMax = a.segMax + static_cast<long long>(b) * a.maxSegs + static_cast<long long>(j) * a.segsPerBlock;
    float *segSum = a.segSum + static_cast<long long>(b) * a.maxSegs + static_cast<long long>(j) * a.segsPerBlock;
    float mb = -INFINITY;
    int k = -1;
    RunMax visit;
    auto mark = [&](int off, float s) {
        if (off % kSeg == 0) {
            if (k >= 0) {
                segMax[k] = visit.m;
                mb = fmaxf(mb, visit.m);
            }
            ++k;
            visit.m = -INFINITY;
            segSum[k] = s;
        }
    };
    mms_main(x, L, start, end, a.W, sum0, visit, mark);
    segMax[k] = visit.m;   // start < end: the first loop step marked checkpoint 0
    a.blockMax[static_cast<long long>(b) * a.maxBlocks + j] = fmaxf(mb, visit.m);
}

// Pass 2: one workgroup per clip reduces pass 1's records to the cut-off (unless the reference
// power fixes it), finds the first and the last reset block holding a hit, in them the first and
// the last checkpoint span holding one, and reruns the recurrence over only those two spans from
// their recorded sums.
__global__ void __launch_bounds__(kPass2Threads) nsr_region_kernel(NsrArgs a)
{
    const int b = blockIdx.x;
    const int L = clip_len(a, b);
    const int nb = blocks_of(L, a.R);
    __shared__ float sMax[kPass2Threads];
    __shared__ int sFirstBlk, sLastBlk, sFirst, sLast, sBegin, sEnd;
    if (threadIdx.x == 0) {
        sFirstBlk = 0x7fffffff;
        sLastBlk = -1;
        sFirst = 0x7fffffff;
        sLast = -1;
        sBegin = L;
        sEnd = -1;
    }
    __syncthreads();

    const int R = a.R <= 0 ? L : a.R;
    const float mf = a.meanFactor;
    const float *bm = a.blockMax + static_cast<long long>(b) * a.maxBlocks;
    float m = -INFINITY;
    for (int j = threadIdx.x; j < nb; j += kPass2Threads) m = fmaxf(m, bm[j]);
    sMax[threadIdx.x] = m;
    __syncthreads();
    for (int s = kPass2Threads / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) sMax[threadIdx.x] = fmaxf(sMax[threadIdx.x], sMax[threadIdx.x + s]);
        __syncthreads();
    }
    // the reference power, else the largest mms, times the cut-off ratio
    const float cut = a.refPower != 0.0f ? a.refPower * a.cutOff : (sMax[0] * mf) * a.cutOff;
    // the first and the last reset block holding a hit, then the first checkpoint span of the
    // one and the last of the other holding a hit
    for (int j = threadIdx.x; j < nb; j += kPass2Threads) {
        if (bm[j] * mf >= cut) {
            atomicMin(&sFirstBlk, j);
            atomicMax(&sLastBlk, j);
        }
    }
    __syncthreads();
    if (sLastBlk >= 0) {
        const float *sm = a.segMax + static_cast<long long>(b) * a.maxSegs;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int j = h == 0 ? sFirstBlk : sLastBlk;
            const long long blockEnd = min(static_cast<long long>(L), static_cast<long long>(j) * R + R);
            const int segs = static_cast<int>((blockEnd - static_cast<long long>(j) * R + kSeg - 1) / kSeg);
            for (int k = threadIdx.x; k < segs; k += kPass2Threads) {
                const int g = j * a.segsPerBlock + k;
                if (sm[g] * mf >= cut) {
                    if (h == 0) atomicMin(&sFirst, g);
                    else atomicMax(&sLast, g);
                }
            }
        }
        __syncthreads();
        // the squares of the two spans' samples and trailing samples x[p - W + 1] go to LDS
        // (0 where p < W - 1: x - 0 is x, the HOST's skipped subtraction); one lane per span
        // runs the additions in order and keeps every running sum; then all threads search
        __shared__ float sQ[2][kSeg], sR[2][kSeg], sS[2][kSeg];
        const float *x = a.src + b * a.nStride;
        int s0[2], n[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int g = h == 0 ? sFirst : sLast;
            const int j = g / a.segsPerBlock;
            s0[h] = j * R + (g - j * a.segsPerBlock) * kSeg;
            const long long e0 = min(static_cast<long long>(L),
                                     min(static_cast<long long>(s0[h]) + kSeg, static_cast<long long>(j) * R + R));
            n[h] = static_cast<int>(e0 - s0[h]);
            for (int i = threadIdx.x; i < n[h]; i += kPass2Threads) {
                const int t = s0[h] + i - a.W + 1;
                const float v = x[s0[h] + i];
                const float w = t >= 0 ? x[t] : 0.0f;
                sQ[h][i] = v * v;
                sR[h][i] = w * w;
            }
        }
        __syncthreads();
        if (threadIdx.x == 0 || threadIdx.x == kWave) {
            const int h = threadIdx.x == 0 ? 0 : 1;
            float sum = a.segSum[static_cast<long long>(b) * a.maxSegs + (h == 0 ? sFirst : sLast)];
            const int nh = n[h];
#pragma unroll 8
            for (int i = 0; i < nh; i++) {
                sum = sum + sQ[h][i];
                sS[h][i] = sum;
                sum = sum - sR[h][i];
            }
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; h++) {
            for (int i = threadIdx.x; i < n[h]; i += kPass2Threads) {
                if (sS[h][i] * mf >= cut) {
                    if (h == 0) atomicMin(&sBegin, s0[h] + i);
                    else atomicMax(&sEnd, s0[h] + i);
                }
            }
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int begin = 0, length = 0;
        if (L > 0 && sEnd >= 0 && sBegin <= sEnd) {
            begin = sBegin;
            length = sEnd - sBegin + 1;
            if (begin != 0) {  // HOST :179-184
                const int nbgn = max(begin - (a.W - 1), 0);
                length += begin - nbgn;
                begin = nbgn;
            }
        }
        a.begin[b] = begin;
        a.length[b] = length;
    }
}

}  // namespace
}  // namespace rppa

// Validation follows rppt_tensor_audio_augmentations.cpp:332-369; windowLength < 1 and a
// resetInterval of 0 or below -1 (which make the HOST loop divide by zero or never advance) are
// rejected with RPP_ERROR_INVALID_ARGUMENTS.
RPPA_EXPORT RppStatus rppt_non_silent_region_detection_gpu(RppPtr_t srcPtr, RpptDescPtr srcDescPtr,
                                                           Rpp32s *srcLengthTensor, Rpp32s *detectedIndexTensor,
                                                           Rpp32s *detectionLengthTensor, Rpp32f cutOffDB,
                                                           Rpp32s windowLength, Rpp32f referencePower,
                                                           Rpp32s resetInterval, rppHandle_t rppHandle)
{
    if (!rppHandle || !srcDescPtr) return RPP_ERROR_INVALID_ARGUMENTS;
    if (srcDescPtr->numDims - 1 != 1) return RPP_ERROR_INVALID_SRC_DIMS;
    if (srcDescPtr->dataType != F32) return RPP_ERROR_NOT_IMPLEMENTED;
    if (!srcPtr || !srcLengthTensor || !detectedIndexTensor || !detectionLengthTensor) return RPP_ERROR_INVALID_ARGUMENTS;
    if (windowLength < 1 || resetInterval == 0 || resetInterval < -1) return RPP_ERROR_INVALID_ARGUMENTS;
    const int B = static_cast<int>(srcDescPtr->n);
    if (B == 0) return RPP_SUCCESS;
    const long long nStride = srcDescPtr->strides.nStride;
    if (nStride < 1 || nStride > 0x7fffffffLL) return RPP_ERROR_INVALID_ARGUMENTS;

    rppa::NsrArgs a{};
    a.src = static_cast<const float *>(srcPtr);
    a.nStride = nStride;
    a.len = srcLengthTensor;
    a.W = static_cast<int>(std::min<long long>(windowLength, nStride + 1));
    a.meanFactor = 1.0f / static_cast<float>(windowLength);
    a.R = resetInterval;
    a.maxBlocks = resetInterval <= 0 ? 1 : static_cast<int>((nStride + resetInterval - 1) / resetInterval);
    a.cutOff = std::pow(10.0f, cutOffDB * 0.1f);
    a.refPower = referencePower;
    a.begin = detectedIndexTensor;
    a.length = detectionLengthTensor;
    const bool stream = static_cast<long long>(B) * nStride * 4 < (1LL << 31);   // a buffer resource's 32-bit offsets
    a.srcBytes = stream ? static_cast<int>(static_cast<long long>(B) * nStride * 4) : 0;
    a.segsPerBlock = static_cast<int>(((resetInterval <= 0 ? nStride : resetInterval) + rppa::kSeg - 1) / rppa::kSeg);
    a.maxSegs = resetInterval <= 0 ? a.segsPerBlock : a.maxBlocks * a.segsPerBlock;
    const size_t cells = static_cast<size_t>(B) * a.maxBlocks;
    const size_t segCells = static_cast<size_t>(B) * a.maxSegs;
    char *ws = static_cast<char *>(rppa::workspace(rppHandle, segCells * 8 + cells * 4));
    if (!ws) return RPP_ERROR_NOT_ENOUGH_MEMORY;
    a.segMax = reinterpret_cast<float *>(ws);
    a.segSum = reinterpret_cast<float *>(ws + segCells * 4);
    a.blockMax = reinterpret_cast<float *>(ws + segCells * 8);

    if (stream) {
        const bool planned = B <= rppa::kPlanned && a.maxBlocks > 1;
        const unsigned g1 = static_cast<unsigned>((cells + rppa::kRows - 1) / rppa::kRows);
        const size_t bytes = planned ? sizeof(int) * (B + 1 + rppa::kStreamThreads / rppa::kWave) : 0;
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(&rppa::nsr_blocks_stream_kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
        hipLaunchKernelGGL(rppa::nsr_blocks_stream_kernel, dim3(g1), dim3(rppa::kStreamThreads), bytes, rppHandle->stream, a, B, planned ? 1 : 0);
    } else {
        const unsigned g1 = static_cast<unsigned>((cells + rppa::kPass1Rows - 1) / rppa::kPass1Rows);
        hipLaunchKernelGGL(rppa::nsr_blocks_kernel, dim3(g1), dim3(rppa::kPass1Threads), 0, rppHandle->stream, a, B);
    }
    RPPA_HIP(hipGetLastError());
    hipLaunchKernelGGL(rppa::nsr_region_kernel, dim3(B), dim3(rppa::kPass2Threads), 0, rppHandle->stream, a);
    RPPA_HIP(hipGetLastError());
    return RPP_SUCCESS;
}
