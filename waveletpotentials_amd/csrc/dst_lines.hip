// DST-I passes with one line per lane, FP32, lines of n = 2^LOGM - 1 samples,
// LOGM = 2..8 (sweep.hip holds the algorithm's derivation and the passes of the
// other lengths).
//
// A lane holds its whole line in registers: the samples are folded into the
// half-length complex sequence in place, transformed by an FFT that is unrolled
// completely (every index, twiddle and sine weight is an immediate, the
// bit-reversed order costs nothing) and turned into the sine coefficients in
// place, without an LDS round trip or a barrier.  About 5400 VALU instructions for
// 255 samples, 9 us of a SIMD's time, against a pass's memory time of about 28
// us at 255^3; the half-wavefront-per-line transform in LDS (sweep.hip) takes 95
// us, all LDS latency.  One wavefront per SIMD (512 registers), which is also
// what 255^2 lines give.
//
// Strided lines (x and z axes): each load and store moves a row of 64
// consecutive floats.  Contiguous lines (y): 64 lines are one contiguous block,
// copied through LDS as it lies; n is odd, so the lanes' walks along their lines
// hit every bank once.
//
// The odd outputs are a running sum over the line; it is accumulated in FP64,
// since a sequential FP32 sum of 128 terms would lose what the tree-shaped scan
// of the LDS kernel keeps.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "whhd_internal.h"

namespace whhd {
namespace dstl {

template <int I>
using ic = std::integral_constant<int, I>;
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(ic<B>{});
        static_for<B + 1, E>(f);
    }
}

// sin(pi a / b) at compile time: reduced to [0, pi / 4], Taylor series in FP64
constexpr double kPi = 3.14159265358979323846;
constexpr double series_sin(double x) {
    double t = x, s = x;
    for (int k = 1; k < 14; ++k) {
        t *= -x * x / ((2 * k) * (2 * k + 1));
        s += t;
    }
    return s;
}
constexpr double series_cos(double x) {
    double t = 1.0, s = 1.0;
    for (int k = 1; k < 14; ++k) {
        t *= -x * x / ((2 * k - 1) * (2 * k));
        s += t;
    }
    return s;
}
constexpr double sin_pi(int a, int b) {
    a %= 2 * b;
    if (a < 0) a += 2 * b;
    if (a >= b) return -sin_pi(a - b, b);
    if (2 * a > b) a = b - a;
    return 4 * a <= b ? series_sin(kPi * a / b) : series_cos(kPi * (b - 2 * a) / (2 * b));
}
constexpr double cos_pi(int a, int b) { return sin_pi(2 * a + b, 2 * b); }

constexpr int bitrev(int v, int bits) {
    int r = 0;
    for (int i = 0; i < bits; ++i) r |= ((v >> i) & 1) << (bits - 1 - i);
    return r;
}

// (r, i) *= e^(-i pi A / B)
template <int A, int B>
__device__ __forceinline__ void mul_w(float& r, float& i) {
    if constexpr (A == 0) {
    } else if constexpr (2 * A == B) {  // -i
        const float t = r;
        r = i;
        i = -t;
    } else {
        constexpr float c = (float)cos_pi(A, B), s = (float)sin_pi(A, B);
        const float t = r * c + i * s;
        i = i * c - r * s;
        r = t;
    }
}

// In-place FFT of P points, decimation in frequency: h[t] = x[2t] + i x[2t + 1];
// point k ends up at bitrev(k).
template <int P, int LEN>
__device__ __forceinline__ void fft(float* x) {
    if constexpr (LEN >= 2) {
        constexpr int half = LEN / 2;
        static_for<0, P / LEN>([&](auto bi) {
            static_for<0, half>([&](auto ji) {
                constexpr int a = decltype(bi)::value * LEN + decltype(ji)::value, b = a + half;
                const float ar = x[2 * a], ai = x[2 * a + 1], br = x[2 * b], bi_ = x[2 * b + 1];
                x[2 * a] = ar + br;
                x[2 * a + 1] = ai + bi_;
                float dr = ar - br, di = ai - bi_;
                mul_w<2 * decltype(ji)::value, LEN>(dr, di);
                x[2 * b] = dr;
                x[2 * b + 1] = di;
            });
        });
        fft<P, LEN / 2>(x);
    }
}

// x[1..M-1]: the line; on return x[j] = c2 * 2 F_j, the DST-I coefficient j - 1 for
// c2 = sqrt(2 / M) / 2.
template <int LOGM>
__device__ __forceinline__ void dst_line(float* x, float c2) {
    constexpr int M = 1 << LOGM, P = M / 2;
    // g_m, g_{M-m} = sin(pi m / M) (f_m + f_{M-m}) +- (f_m - f_{M-m}) / 2; g_0 = 0, g_P = 2 f_P
    x[0] = 0.f;
    static_for<1, P>([&](auto mi) {
        constexpr int m = decltype(mi)::value;
        constexpr float s = (float)sin_pi(m, M);
        const float a = s * (x[m] + x[M - m]), b = 0.5f * (x[m] - x[M - m]);
        x[m] = a + b;
        x[M - m] = a - b;
    });
    x[P] = 2.f * x[P];
    fft<P, P>(x);
    // 2 G_k = E + w O, 2 G_{P-k} = conj(E - w O), E = H_k + conj H_{P-k}, O = (H_k - conj
    // H_{P-k}) / i, w = e^{-2 pi i k / M}; Re in place of H_k's real part, Im of the other
    static_for<1, (P + 1) / 2>([&](auto ki) {
        constexpr int k = decltype(ki)::value, a = bitrev(k, LOGM - 1), b = bitrev(P - k, LOGM - 1);
        const float er = x[2 * a] + x[2 * b], ei = x[2 * a + 1] - x[2 * b + 1];
        float wr = x[2 * a + 1] + x[2 * b + 1], wi = x[2 * b] - x[2 * a];
        mul_w<2 * k, M>(wr, wi);
        x[2 * a] = er + wr;
        x[2 * a + 1] = ei + wi;
        x[2 * b] = er - wr;
        x[2 * b + 1] = wi - ei;
    });
    {   // k = 0: G_0 = Re H_0 + Im H_0; k = P / 2: w = -i, G = conj H
        const float g0 = x[0] + x[1];
        x[0] = g0;  // 2 F_1 = Re G_0: half of 2 Re G_0
        if constexpr (P >= 2) {
            constexpr int a = bitrev(P / 2, LOGM - 1);
            x[2 * a] = 2.f * x[2 * a];
            x[2 * a + 1] = -2.f * x[2 * a + 1];
        }
    }
    // F_{2k+1} = F_{2k-1} + Re G_k, F_{2k} = -Im G_k, in natural order
    float y[M];
    double run = 0.0;
    static_for<0, P>([&](auto ki) {
        constexpr int k = decltype(ki)::value, a = bitrev(k, LOGM - 1);
        run += (double)x[2 * a];
        y[2 * k + 1] = c2 * (float)run;
        if constexpr (k > 0) y[2 * k] = -c2 * x[2 * a + 1];
    });
    static_for<1, M>([&](auto j) { x[decltype(j)::value] = y[decltype(j)::value]; });
}

struct Args {
    float* out;
    const float* in;
    uint32_t lines, n_inner, s_inner, s_outer, step;
    float c2;
    // reps = 2: transform, divide by lam_q[li / lam_div] + lam_r[li % lam_div] + lam_s[j], transform
    const float *lam_q, *lam_r, *lam_s;
    uint32_t lam_div;
    int scale, reps;
};

template <int LOGM, bool CONTIG>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1, 2))) dst_lines_kernel(Args a) {
    constexpr int M = 1 << LOGM, N = M - 1;
    // contiguous runs of tiles per XCD, see sweep.hip
    const unsigned nwg = gridDim.x, r8 = blockIdx.x % 8u, q8 = blockIdx.x / 8u;
    const unsigned tile = r8 * (nwg / 8u) + (r8 < nwg % 8u ? r8 : nwg % 8u) + q8;
    const int lane = threadIdx.x;
    const uint32_t first = tile * 64u;
    const bool ok = first + lane < a.lines;
    const uint32_t li = ok ? first + lane : first;
    float x[M];
    uint32_t base = 0;
    [[maybe_unused]] float* lds = nullptr;
    [[maybe_unused]] uint32_t elems = 0;
    if constexpr (CONTIG) {
        extern __shared__ __attribute__((aligned(16))) float dst_lds[];
        lds = dst_lds;
        elems = min(64u, a.lines - first) * N;
        const float* src = a.in + (size_t)first * N;  // 16-byte aligned: 64 N floats a tile
        const uint32_t quads = elems / 4;
#pragma unroll 16
        for (uint32_t e = lane; e < quads; e += 64) ((float4*)lds)[e] = ((const float4*)src)[e];
        if (4 * quads + lane < elems) lds[4 * quads + lane] = src[4 * quads + lane];
        __syncthreads();
        const float* row = lds + (ok ? lane : 0) * N;
        static_for<1, M>([&](auto j) { x[decltype(j)::value] = row[decltype(j)::value - 1]; });
    } else {
        const uint32_t o = li / a.n_inner, i = li - o * a.n_inner;
        base = i * a.s_inner + o * a.s_outer;
        const float* src = a.in + base;
        static_for<1, M>([&](auto j) { x[decltype(j)::value] = src[(size_t)(decltype(j)::value - 1) * a.step]; });
    }
    dst_line<LOGM>(x, a.c2);
    if (a.scale) {
        const uint32_t q = li / a.lam_div;
        const float sum = a.lam_q[q] + a.lam_r[li - q * a.lam_div];
        static_for<1, M>([&](auto j) {
            // reciprocal (within 1 ulp) instead of an IEEE division
            x[decltype(j)::value] *= __builtin_amdgcn_rcpf(sum + a.lam_s[decltype(j)::value - 1]);
        });
    }
    if (a.reps == 2) dst_line<LOGM>(x, a.c2);
    if constexpr (CONTIG) {
        float* row = lds + lane * N;
        if (ok) static_for<1, M>([&](auto j) { row[decltype(j)::value - 1] = x[decltype(j)::value]; });
        __syncthreads();
        float* dst = a.out + (size_t)first * N;
        const uint32_t quads = elems / 4;
#pragma unroll 16
        for (uint32_t e = lane; e < quads; e += 64) ((float4*)dst)[e] = ((const float4*)lds)[e];
        if (4 * quads + lane < elems) dst[4 * quads + lane] = lds[4 * quads + lane];
    } else if (ok) {
        float* dst = a.out + base;
        static_for<1, M>([&](auto j) { dst[(size_t)(decltype(j)::value - 1) * a.step] = x[decltype(j)::value]; });
    }
}

}  // namespace dstl

// One DST-I pass of `lines` lines of 2^logm - 1 samples, as dst_fft_kernel's
// arguments describe them; false where no kernel applies, or where dst_fft_kernel's
// half-wavefront per line is faster: a lane's 255 samples take 13 us however few the
// lines are (us a pass, line per lane against it: strided, up to 4098 lines +4, 8194
// -1.5, 16386 -10; contiguous, up to 4098 lines +6, 8194 +2, 16386 -7; a planar 255^2
// solve 65 against 41).  Shorter lines are faster a line per lane at every count
// (127 samples 16 lines -3, 63 samples -7, contiguous -6 and -13).
bool dst_lines(int logm, bool contig, float* out, const float* in, int64_t lines, int64_t n_inner,
               int64_t s_inner, int64_t s_outer, int64_t step, float c, const float* lam_q,
               const float* lam_r, const float* lam_s, int64_t lam_div, int reps, hipStream_t s) {
    const int64_t n = (1 << logm) - 1;
    if (logm == 8 && lines < (contig ? 12288 : 8192)) return false;
    if (logm < 2 || logm > 8 || lines < 1 || lines * n >= (int64_t)1 << 31) return false;
    if (contig && (((uintptr_t)in | (uintptr_t)out) & 15)) return false;  // 16-byte copies
    const dstl::Args a{out, in, (uint32_t)lines, (uint32_t)n_inner, (uint32_t)s_inner, (uint32_t)s_outer,
                       (uint32_t)step, 0.5f * c, lam_q, lam_r, lam_s, (uint32_t)lam_div, lam_s != nullptr, reps};
    const dim3 grid((unsigned)((lines + 63) / 64)), block(64);
    const size_t lds = contig ? 64 * n * sizeof(float) : 0;
#define WHHD_DSTL(L)                                                                                   \
    case L:                                                                                            \
        if (contig) hipLaunchKernelGGL((dstl::dst_lines_kernel<L, true>), grid, block, lds, s, a);     \
        else hipLaunchKernelGGL((dstl::dst_lines_kernel<L, false>), grid, block, 0, s, a);             \
        return true;
    switch (logm) {
        WHHD_DSTL(2) WHHD_DSTL(3) WHHD_DSTL(4) WHHD_DSTL(5) WHHD_DSTL(6) WHHD_DSTL(7) WHHD_DSTL(8)
    }
#undef WHHD_DSTL
    return false;
}

}  // namespace whhd
