// log2_math.hpp -- FP32 log2 through FP64, rounded once: the to_decibels kernel and the FP32 fused
// launch share it, so both give the same bits.
#pragma once

#include <hip/hip_runtime.h>

namespace rppa {

// For i = 0 .. 64: c, the FP32 value nearest 1 / (1/2 + i / 128), and -log2 c.
struct alignas(16) Log2Entry {
    double log;
    float c;
};
__device__ const Log2Entry kLog2[65] = {
    {-1.0, 2.0f}, {-0.97763218831516, 1.9692307710647583f}, {-0.9556059236372086, 1.9393939971923828f},
    {-0.9339107759518657, 1.9104477167129517f}, {-0.9125371641241184, 1.8823529481887817f}, {-0.8914755700941199, 1.8550724983215332f},
    {-0.8707169911167203, 1.8285714387893677f}, {-0.8502528536230285, 1.8028168678283691f}, {-0.8300750093066033, 1.7777777910232544f},
    {-0.8101754303710671, 1.7534246444702148f}, {-0.7905466693050257, 1.7297297716140747f}, {-0.7711813444380946, 1.7066667079925537f},
    {-0.7520724973053301, 1.6842105388641357f}, {-0.7332134579614842, 1.6623376607894897f}, {-0.7145977999483539, 1.6410256624221802f},
    {-0.696219288100487, 1.6202532052993774f}, {-0.6780719266104689, 1.600000023841858f}, {-0.6601500078642909, 1.580246925354004f},
    {-0.6424479416373369, 1.5609755516052246f}, {-0.6249605149084958, 1.5421686172485352f}, {-0.6076826040935287, 1.523809552192688f},
    {-0.5906090920782017, 1.5058823823928833f}, {-0.5737352399234442, 1.4883720874786377f}, {-0.5570564987768138, 1.471264362335205f},
    {-0.5405684243583648, 1.454545497894287f}, {-0.5242665838133612, 1.4382022619247437f}, {-0.5081469386043008, 1.4222222566604614f},
    {-0.4922053960788937, 1.4065934419631958f}, {-0.47643807081527606, 1.39130437374115f}, {-0.4608411875483541, 1.376344084739685f},
    {-0.44541110263947026, 1.3617020845413208f}, {-0.430144453475316, 1.3473684787750244f}, {-0.4150375422745059, 1.3333333730697632f},
    {-0.40008711347359444, 1.3195875883102417f}, {-0.3852901263252734, 1.3061224222183228f}, {-0.37064337857677593, 1.2929292917251587f},
    {-0.3561437779785279, 1.2799999713897705f}, {-0.3417884944067593, 1.2673267126083374f}, {-0.32757470908585296, 1.2549020051956177f},
    {-0.3134994862529262, 1.2427184581756592f}, {-0.2995603356034852, 1.2307692766189575f}, {-0.2857545374220692, 1.2190476655960083f},
    {-0.27207956693463203, 1.2075471878051758f}, {-0.2585329679159607, 1.1962616443634033f}, {-0.2451125085854471, 1.185185194015503f},
    {-0.23181561341680718, 1.174311876296997f}, {-0.21864024079244804, 1.163636326789856f}, {-0.20558416858386958, 1.1531531810760498f},
    {-0.1926451424358885, 1.1428571939468384f}, {-0.17982103221035445, 1.1327433586120605f}, {-0.16710999658417397, 1.1228070259094238f},
    {-0.15450988321851475, 1.1130434274673462f}, {-0.14201899949797003, 1.1034482717514038f}, {-0.1296353516281601, 1.0940171480178833f},
    {-0.11735695332538766, 1.0847457647323608f}, {-0.10518231059084988, 1.0756303071975708f}, {-0.09310947963388926, 1.0666667222976685f},
    {-0.08113670226275353, 1.0578511953353882f}, {-0.06926258182024388, 1.049180269241333f}, {-0.05748544091618073, 1.0406503677368164f},
    {-0.04580364661746143, 1.0322580337524414f}, {-0.03421578386224878, 1.0240000486373901f}, {-0.022720159804177638, 1.0158730745315552f},
    {-0.011315307853376297, 1.0078740119934082f}, {0.0, 1.0f}};

// The table where it lies, and its copy in LDS where a kernel has room for it: there a wave's different entries meet at
// most two or three to a bank (65 doubles are 130 words over 64 banks: entries i and i + 32 share theirs; of the floats
// only the first and the last do), while from memory they are 64 separate 16-byte reads (to_decibels on the spectra of 128
// clips of 80 bands: 22 us from memory, 17 us from LDS).
struct Log2Global {
    __device__ double log(unsigned i) const { return kLog2[i].log; }
    __device__ float c(unsigned i) const { return kLog2[i].c; }
};
struct Log2Lds {
    double logs[65];
    float cs[65];
    __device__ void fill()   // by the whole block (65 threads at least); ends with a barrier
    {
        if (threadIdx.x < 65) set(threadIdx.x, kLog2[threadIdx.x]);
        __syncthreads();
    }
    __device__ void set(int i, const Log2Entry &e)
    {
        logs[i] = e.log;
        cs[i] = e.c;
    }
    __device__ double log(unsigned i) const { return logs[i]; }
    __device__ float c(unsigned i) const { return cs[i]; }
};

// log2(x) for x > 0 (subnormal and infinite x included).  With x = f 2^e, f in [1/2, 1), and c the reciprocal of the
// nearest of 65 points of that interval: log2 x = (e - log2 c) + log2(1 + r), r = f c - 1 (exact), |r| <= 2^-7, by the
// series to r^7.  Around x = 1 the points are 1/2 and 1 themselves, where c is exact and e - log2 c is 0, so the
// relative error stays below 2^-49 and the rounding to FP32 differs from the correctly rounded value only within
// 2^-25 ulp of a tie.  A dozen FP64 operations against some 30 (a division and a series to the 19th power) without a
// table and 90 of the library's log2.
template <typename Table>
__device__ __forceinline__ float log2_rn(float x, const Table &t)
{
    const float f = __builtin_amdgcn_frexp_mantf(x);
    const int e = __builtin_amdgcn_frexp_expf(x);
    const unsigned i = min(static_cast<unsigned>(fmaf(f, 128.0f, -63.5f)), 64u);   // (min: an infinite x)
    const double r = fma(static_cast<double>(f), static_cast<double>(t.c(i)), -1.0);
    double p = 0.2060992915555662;
    p = fma(p, r, -0.2404491734814939);
    p = fma(p, r, 0.28853900817779266);
    p = fma(p, r, -0.36067376022224085);
    p = fma(p, r, 0.4808983469629878);
    p = fma(p, r, -0.7213475204444817);
    p = fma(p, r, 1.4426950408889634);
    const double v = fma(p, r, static_cast<double>(e) + t.log(i));
    return x < __builtin_inff() ? static_cast<float>(v) : x;
}

}  // namespace rppa
