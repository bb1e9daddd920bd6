// fft_real.hpp -- power spectra of real FP32 frames by FFT, shared by the spectrogram and the fused FP32
// log-mel kernels so both give the same bits.
//
// A frame of N real samples is packed as M = N/2 complex ones, z[n] = w x[2n] + i w x[2n+1], and
// transformed as M = R1 x R2 (R1 <= R2) by R1 lanes ("a group"; a wave holds 64 / R1 groups, one
// frame each):
//   pass 1  lane l runs the R1-point FFTs of the columns n2 = l, l + R1, ..., each over
//           z[R2 n1 + n2], and multiplies output k1 by exp(-2 pi i n2 k1 / M);
//   turn    a transpose through the wave's own LDS (real parts, then imaginary parts, so one plane
//           of M values is enough), after which lane k1 holds all n2 of its k1;
//   pass 2  lane k1 runs one R2-point FFT: Z[k1 + R1 k2] for every k2;
//   split   X[k] = E + W^k O and X[M-k] = conj(E - W^k O), E and O from Z[k] and Z[M-k].  Bin M-k
//           belongs to lane R1 - k1 (itself for k1 = 0), so half of each lane's values are
//           exchanged once and every pair is formed once.
// The factor 1/2 of E and O is folded into the window table (exact).  Every step of a wave touches
// only its own LDS, so no workgroup barrier is needed up to the power values.
//
// The arithmetic is FP64, at about 1.6 times the issue time of FP32 here (without packed FP32), and each power value
// is rounded once.  In FP32 the transform's rounding is white noise at 2^-24 of the frame's norm: a quarter of the dense FP32
// contraction's error in the spectrum's norm, but twice its error in the dB of pre-emphasised music (bins 80 dB
// below the frame, whose dense partial sums stay as small as the bins are); in FP64 both are below it (24 clips of 2-10 s at 44.1
// kHz, nfft 1024, 128 filters: dB off by 1.9e-6 of its norm dense, 3.6e-6 in FP32, 1.7e-6 in FP64).
#pragma once

#include "common.hpp"

namespace rppa {

// cos(2 pi j / 64), j = 0 .. 16
__device__ constexpr double kCos64[17] = {
    1.0, 0.99518472667219693, 0.98078528040323043, 0.95694033573220882, 0.92387953251128674,
    0.88192126434835505, 0.83146961230254524, 0.77301045336273699, 0.70710678118654757,
    0.63439328416364549, 0.55557023301960229, 0.47139673682599781, 0.38268343236508984,
    0.29028467725446233, 0.19509032201612833, 0.09801714032956077, 0.0};

// exp(-2 pi i j / R) for 0 <= j < R / 2, R a power of two up to 64
template <int R>
__device__ constexpr double tw_cos(int j)
{
    const int q = j * (64 / R);   // 0 .. 31
    return q <= 16 ? kCos64[q] : -kCos64[32 - q];
}
template <int R>
__device__ constexpr double tw_sin(int j)   // sin(2 pi j / R)
{
    const int q = j * (64 / R);
    return q <= 16 ? kCos64[16 - q] : kCos64[q - 16];
}

template <int R>
__device__ constexpr int bit_rev(int i)
{
    int r = 0;
    for (int b = 1; b < R; b <<= 1) {
        r = (r << 1) | (i & 1);
        i >>= 1;
    }
    return r;
}

// One level of a radix-2 decimation-in-frequency FFT of length LEN at v[BASE ..], then its halves.
template <int LEN, int BASE, int R>
__device__ __forceinline__ void fft_level(double (&re)[R], double (&im)[R])
{
    if constexpr (LEN > 1) {
#pragma unroll
        for (int j = 0; j < LEN / 2; j++) {
            const int p = BASE + j, q = p + LEN / 2;
            const double ar = re[p], ai = im[p], br = re[q], bi = im[q];
            re[p] = ar + br;
            im[p] = ai + bi;
            const double dr = ar - br, di = ai - bi;
            if (j == 0) {
                re[q] = dr;
                im[q] = di;
            } else if (4 * j == LEN) {          // -i
                re[q] = di;
                im[q] = -dr;
            } else if (8 * j == LEN) {          // (1 - i) / sqrt 2
                re[q] = (di + dr) * kCos64[8];
                im[q] = (di - dr) * kCos64[8];
            } else if (8 * j == 3 * LEN) {      // (-1 - i) / sqrt 2
                re[q] = (di - dr) * kCos64[8];
                im[q] = (di + dr) * -kCos64[8];
            } else {
                const double c = tw_cos<LEN>(j), s = tw_sin<LEN>(j);
                re[q] = fma(di, s, dr * c);
                im[q] = fma(-dr, s, di * c);
            }
        }
        fft_level<LEN / 2, BASE, R>(re, im);
        fft_level<LEN / 2, BASE + LEN / 2, R>(re, im);
    }
}

// R-point complex FFT in registers; output k is left in element bit_rev<R>(k).
template <int R>
__device__ __forceinline__ void fft_regs(double (&re)[R], double (&im)[R])
{
    fft_level<R, 0, R>(re, im);
}

constexpr bool rfft_supported(int nfft)
{
    return nfft == 64 || nfft == 128 || nfft == 256 || nfft == 512 || nfft == 1024 || nfft == 2048;
}

// Tables of one (nfft, W, window) in the order the lanes read them, 16 bytes at a time (l: lane in its group): the
// halved FP32 window, zero past W, [j][n1 / 2][l][4] = pairs n = R2 n1 + R1 j + l of n1, n1 + 1; in FP64 the twiddles
// (cos, -sin)(2 pi n2 k1 / M), [j][k1][l][2], n2 = R1 j + l, and the split factors (cos, sin)(2 pi k / N), [k2][l][2],
// k = l + R1 k2 < M / 2.
constexpr size_t rfft_table_floats(int nfft) { return static_cast<size_t>(nfft) * 4; }

template <int N>
struct RealFft {
    static constexpr int M = N / 2;
    static constexpr int R1 = N <= 64 ? 4 : N <= 256 ? 8 : N <= 1024 ? 16 : 32;
    static constexpr int R2 = M / R1;
    static constexpr int kSub = R2 / R1;            // pass-1 columns per lane
    static constexpr int kGroups = kWave / R1;      // frames per wave
    // turn buffer, in doubles: row k1 of R2 values padded to keep 16-byte alignment, groups offset by R1
    // values (mod 32), so the 8-byte writes of a wave fall on all 64 banks and the reads are 16 bytes wide
    static constexpr int kRow = R2 + 2;
    static constexpr int kGroupPitch = (R1 * kRow + 31) / 32 * 32 + R1;
    static constexpr int kTurnFloats = 2 * kGroups * kGroupPitch;   // LDS floats per wave

    static_assert(R1 * R2 == M && R2 % R1 == 0, "M = R1 x R2");

    // The tables' address for one frame: the compiler must not keep the tables in registers across frames
    // (they would take more than the data).
    static __device__ __forceinline__ const double *per_frame(const double *tab) { return N > 256 ? per_call(tab) : tab; }
    static __device__ __forceinline__ const double *per_call(const double *tab)
    {
        unsigned zero = 0;   // (an opaque offset: an opaque pointer would lose its address space)
        __asm__ volatile("" : "+s"(zero));
        return tab + zero;
    }

    // LDS written by this wave is read by its other lanes after this
    static __device__ __forceinline__ void wave_sync()
    {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }

    // Samples past the window (2n >= W) do not count, whatever they are: the rows that reach past it
    // are masked, one uniform branch per row of columns (the asm keeps it a branch: turned into
    // selects it is a hundred scalar mask operations per frame).
    static __device__ __forceinline__ void mask_window(int W, int l, float (&zr)[kSub][R1], float (&zi)[kSub][R1])
    {
#pragma unroll
        for (int n1 = 0; n1 < R1; n1++)
            if (2 * R2 * (n1 + 1) > W) {
                __asm__ volatile("" : "+v"(l));
#pragma unroll
                for (int j = 0; j < kSub; j++) {
                    const int t = 2 * (R2 * n1 + R1 * j + l);
                    zr[j][n1] = t < W ? zr[j][n1] : 0.0f;
                    zi[j][n1] = t + 1 < W ? zi[j][n1] : 0.0f;
                }
            }
    }

    // One frame per group up to pass 2.  zr/zi[j][n1] hold the frame's samples 2n and 2n + 1, n = R2 n1 +
    // R1 j + l (l the lane in its group), zero past the window; Z[l + R1 k2] is left in element
    // bit_rev<R2>(k2) of ar/ai.   tab: the tables, turn: the wave's buffer + group * kGroupPitch
    static __device__ __forceinline__ void transform(const double *__restrict__ tab, double *turn, int lane,
                                                     const float (&zr)[kSub][R1], const float (&zi)[kSub][R1],
                                                     double (&ar)[R2], double (&ai)[R2])
    {
        const unsigned l = lane & (R1 - 1);
        const float4 *__restrict__ win = reinterpret_cast<const float4 *>(tab) + l;
        const double2 *__restrict__ tw = reinterpret_cast<const double2 *>(tab + N / 2) + l;
        double yr[kSub][R1], yi[kSub][R1];
#pragma unroll
        for (int j = 0; j < kSub; j++) {
#pragma unroll
            for (int n1 = 0; n1 < R1; n1 += 2) {   // (products of two FP32 values: exact)
                const float4 w = win[(j * R1 + n1) / 2 * R1];
                yr[j][n1] = static_cast<double>(zr[j][n1]) * w.x;
                yi[j][n1] = static_cast<double>(zi[j][n1]) * w.y;
                yr[j][n1 + 1] = static_cast<double>(zr[j][n1 + 1]) * w.z;
                yi[j][n1 + 1] = static_cast<double>(zi[j][n1 + 1]) * w.w;
            }
            fft_regs<R1>(yr[j], yi[j]);
#pragma unroll
            for (int k1 = 1; k1 < R1; k1++) {
                const int q = bit_rev<R1>(k1);
                const double2 t = tw[(j * R1 + k1) * R1];
                const double xr = yr[j][q], xi = yi[j][q];
                yr[j][q] = fma(-xi, t.y, xr * t.x);
                yi[j][q] = fma(xi, t.x, xr * t.y);
            }
        }
        auto turned = [&](const double (&from)[kSub][R1], double (&to)[R2]) {
            wave_sync();
#pragma unroll
            for (int j = 0; j < kSub; j++)
#pragma unroll
                for (int k1 = 0; k1 < R1; k1++) turn[k1 * kRow + j * R1 + l] = from[j][bit_rev<R1>(k1)];
            wave_sync();
#pragma unroll
            for (int n = 0; n < R2; n += 2) {
                const double2 v = *reinterpret_cast<const double2 *>(&turn[l * kRow + n]);
                to[n] = v.x;
                to[n + 1] = v.y;
            }
        };
        turned(yr, ar);
        turned(yi, ai);
        fft_regs<R2>(ar, ai);
    }

    // The split: store(k, v) takes |X_k|^2.
    template <typename Store>
    static __device__ __forceinline__ void power(const double *__restrict__ tab, int lane, const double (&ar)[R2],
                                                 const double (&ai)[R2], const Store &store)
    {
        const unsigned l = lane & (R1 - 1);
        const double2 *__restrict__ split = reinterpret_cast<const double2 *>(tab + N / 2 + N) + l;
        // this lane's k = l + R1 k2 with k2 < R2 / 2 and its mirror M - k, held by lane R1 - l as
        // k2' = R2 - 1 - k2 (by lane 0 itself as R2 - k2)
        const int src = static_cast<int>(((lane & ~(R1 - 1)) | ((R1 - l) & (R1 - 1))) << 2);
        const bool own = l == 0;
        auto from_mirror = [&](double v) {
            const int lo = __builtin_amdgcn_ds_bpermute(src, __double2loint(v));
            const int hi = __builtin_amdgcn_ds_bpermute(src, __double2hiint(v));
            return __hiloint2double(hi, lo);
        };
#pragma unroll
        for (int k2 = 0; k2 < R2 / 2; k2++) {
            const int p = bit_rev<R2>(k2), m = bit_rev<R2>(R2 - 1 - k2), o = bit_rev<R2>((R2 - k2) & (R2 - 1));
            const double br = from_mirror(ar[m]), bi = from_mirror(ai[m]);
            const double c = own ? ar[o] : br, d = own ? ai[o] : bi;
            const double a = ar[p], b = ai[p];
            const double2 w = split[k2 * R1];
            const double er = a + c, ei = b - d, orr = b + d, oi = c - a;
            const double tr = fma(w.y, oi, w.x * orr), ti = fma(-w.y, orr, w.x * oi);
            const double xr = er + tr, xi = ei + ti, yr = er - tr, yi = ei - ti;
            store(l + R1 * k2, static_cast<float>(fma(xr, xr, xi * xi)));
            store(M - R1 * k2 - l, static_cast<float>(fma(yr, yr, yi * yi)));
        }
        if (own) {   // bin M/2 is its own mirror: X = conj Z (twice the halved window's value)
            const int p = bit_rev<R2>(R2 / 2);
            const double a = 2.0 * ar[p], b = 2.0 * ai[p];
            store(M / 2, static_cast<float>(fma(a, a, b * b)));
        }
    }

    // The wave's frames (bit l of its lanes' ballot: lane 0 of the frame's group) with a sample that is not finite.
    // Z_0 is the plain sum of the windowed pairs, so no such sample leaves it finite, and finite FP32
    // samples cannot overflow it.
    static __device__ __forceinline__ unsigned long long not_finite(int lane, const double (&ar)[R2], const double (&ai)[R2])
    {
        const double inf = __builtin_inf();
        return __ballot((lane & (R1 - 1)) == 0 && !(fabs(ar[0]) < inf && fabs(ai[0]) < inf));
    }

    // The power of those frames after power(): infinite where the contraction of the frame with a bin's cosine and
    // sine columns is, NaN where it holds infinities of both signs or an infinity times a zero of the
    // column, as the dense contraction has it (the transform's products of infinities are NaN in every bin).
    // A NaN sample has made every bin NaN.  sample(g, t): sample t of group g's frame.  One wave, rarely.
    template <typename Sample, typename Store>
    static __device__ __forceinline__ void infinite_power(const double *__restrict__ tab, int W, int lane,
                                                          unsigned long long frames, const Sample &sample, const Store &store)
    {
        const float inf = __builtin_inff();
        // (opaque: nothing of this is computed ahead of the frames' loop, in registers that they would miss)
        __asm__ volatile("" : "+v"(lane));
        __asm__ volatile("" : "+s"(W));
        const float *win = reinterpret_cast<const float *>(per_call(tab));
        for (; frames; frames &= frames - 1) {
            const int g = (__ffsll(frames) - 1) / R1;
            unsigned blocks = 0;   // 64-sample blocks with an infinity
            bool nan = false;
            for (int t0 = 0; t0 < W; t0 += kWave) {
                const float v = t0 + lane < W ? sample(g, t0 + lane) : 0.0f;
                nan = nan || __ballot(v != v) != 0;
                blocks |= __ballot(fabsf(v) == inf) ? 1u << (t0 / kWave) : 0u;
            }
            if (nan) continue;
            for (int k = lane; k - lane <= M; k += kWave) {
                float re = 0.0f, im = 0.0f;
                for (unsigned left = blocks; left; left &= left - 1) {
                    const int t0 = (__ffs(left) - 1) * kWave;
                    const float v = t0 + lane < W ? sample(g, t0 + lane) : 0.0f;
                    for (unsigned long long at = __ballot(fabsf(v) == inf); at; at &= at - 1) {
                        const int i = __ffsll(at) - 1, t = t0 + i, n = t >> 1;
                        const float x = __shfl(v, i);
                        const int n1 = n / R2, j = n % R2 / R1, l = n % R1;
                        const float w = 2.0f * win[((j * R1 + n1) / 2 * R1 + l) * 4 + n1 % 2 * 2 + (t & 1)];
                        // cos and -sin of 2 pi r / N, which alone decide the sign; what FP64 has for their zeros
                        const int r = (k * t) & (N - 1);
                        const float c = r == N / 4 ? 6.1232340e-17f : (r == 3 * N / 4 ? -1.8369702e-16f
                                                                                     : (r < N / 4 || r > 3 * N / 4 ? 1.0f : -1.0f));
                        const float s = r == 0 ? 0.0f : (r == N / 2 ? 1.2246468e-16f : (r < N / 2 ? 1.0f : -1.0f));
                        re = fmaf(x, w * c, re);
                        im = fmaf(x, -(w * s), im);
                    }
                }
                if (k <= M) store(g, k, k == 0 || k == M ? re * re : re * re + im * im);
            }
        }
    }
};

}  // namespace rppa
