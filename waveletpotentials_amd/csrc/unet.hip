// Learned initial guess for the fractional multigrid: a 3-level 3D U-Net
// (16/32/64 channels, 3x3x3 convolutions, ReLU, 2x2x2 average pooling,
// nearest upsampling, concatenated skips) mapping (f, solid level set) to the
// pressure.  No reference counterpart: the reference's multigrid takes its
// initial guess as pre_v (WaveletPotentials/cuMultigridFrac3D.cu:249-258),
// which is where the prediction enters; the plain multigrid remains the solver
// and the judge of convergence.
//
// Everything runs on the device with this file's kernels:
//  * convolutions as implicit GEMMs on the BF16 matrix cores
//    (v_mfma_f32_16x16x32_bf16, FP32 accumulation): rows are voxels, columns
//    output channels, the reduction runs over (tap, input channel); the
//    upsampling and the skip concatenation are folded into the operand reads;
//  * the input gradient is the same kernel with the flipped, transposed
//    weights and the ReLU mask on its output; the weight gradient reduces over
//    voxels from bricks staged transposed in LDS, in slices summed in a fixed order;
//  * pooling, the loss and Adam are element-wise kernels.
// Activations and their gradients are BF16, channels-last ((z, x, y) voxel
// order, channels innermost); master weights, moments and gradients are FP32.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

#include "whhd_internal.h"

namespace whhd {
namespace unet {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

enum { MODE_RELU = 0, MODE_F32 = 1, MODE_GRAD = 2 };

constexpr int kTaps = 27;
constexpr int kIn = 16;  // input channels (f, level set, 14 zero channels)

__host__ __device__ constexpr int kpad(int cin) { return (kTaps * cin + 31) / 32 * 32; }

// Source of a convolution: channels [0, CA) from `a`, at half resolution when
// the layer upsamples it; channels [CA, CA + CB) from `b`; output extents Z, X, Y.
struct ConvSrc {
    const bf16* a;
    const bf16* b;
    int Z, X, Y;
};

struct ConvOut {
    bf16* o1;            // RELU: all CO channels; GRAD: channels [0, split)
    bf16* o2;            // GRAD: channels [split, CO)
    float* of;           // F32: channel 0
    const float* bias;   // RELU, F32
    const bf16* mask;    // GRAD, may be null: o1 is zeroed where this (CO channels) is not positive
    int split;
};

// y = conv3x3x3(x) on a workgroup's brick of BZ x BX x BY voxels and all CO
// channels: D = W X, rows (A operand) output channels, columns (B operand)
// voxels, the reduction over (tap, input channel) in chunks of 32.
//
// The brick's input with its one-voxel halo is staged once in LDS (rows of
// CIN + 8 values: the 16 voxels a fragment reads then start in different banks)
// and every tap reads it there.  The weights come from global memory in
// fragment order (pack_kernel): 1 KB contiguous per wavefront and chunk.  The
// wavefronts split the brick's voxel tiles (WM) and the channel tiles (WN); every
// output is summed by one wavefront over the chunks in their order, whatever the
// split.  The small grids of the lower levels have few voxels, and what bounds them
// is the number of wavefronts a brick and the chip get, not the matrix cores.
// Reading every operand from the caches in each tap, 32 voxels a wavefront, took
// (48^3 network grid) 14.5 us for 16 -> 16 channels, 41 for 48 -> 16 (48^3), 42 for
// 96 -> 32 (24^3) and 42 for 64 -> 64 (12^3); this one 7.0, 14.6, 12.3 and 5.8.  With the
// chunks split over wavefronts too and their sums added through LDS (fewer voxel or
// channel tiles each) the last three took 20, 12.3 and 10.7, and the other order of the
// sum moved single BF16 activations.
template <int CA, int CB, bool UPA, int CO, int MODE, int BZ, int BX, int BY, int WM, int WN>
__global__ void __launch_bounds__(64 * WM * WN) conv3_kernel(ConvSrc s, const bf16* __restrict__ w,
                                                                  ConvOut o) {
    constexpr int CIN = CA + CB;
    static_assert(CIN % 16 == 0 && CA % 8 == 0 && CO % 16 == 0, "channel blocking");
    constexpr int KC = kpad(CIN) / 32;
    constexpr int M = BZ * BX * BY, MT = M / 16, NT = CO / 16, MTW = MT / WM, NTW = NT / WN;
    static_assert(M % 16 == 0 && MT % WM == 0 && NT % WN == 0, "tile split");
    constexpr int HX = BX + 2, HY = BY + 2, HV = (BZ + 2) * HX * HY;
    constexpr int SV = CIN + 8, PV = CIN / 8;
    constexpr int NTHR = 64 * WM * WN, PIECES = HV * PV, PER = (PIECES + NTHR - 1) / NTHR;
    __shared__ __attribute__((aligned(16))) bf16 sm[HV * SV + 8];  // + a zero piece
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave % WM, wn = wave / WM;
    const int m = lane & 15, g = lane >> 4;
    const int by = (s.Y + BY - 1) / BY, bx = (s.X + BX - 1) / BX;
    int bid = blockIdx.x;
    const int y0 = (bid % by) * BY;
    bid /= by;
    const int x0 = (bid % bx) * BX, z0 = (bid / bx) * BZ;
    const int Xh = s.X >> 1, Yh = s.Y >> 1;
    bf16x8 piece[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = tid + i * NTHR;
        const int p = e % PV, hv = e / PV;
        const int zz = z0 + hv / (HX * HY) - 1, xx = x0 + (hv / HY) % HX - 1, yy = y0 + hv % HY - 1;
        const bool in = e < PIECES && zz >= 0 && zz < s.Z && xx >= 0 && xx < s.X && yy >= 0 && yy < s.Y;
        const int ci = 8 * p;
        piece[i] = bf16x8{};
        if (in) {
            if (CB == 0 || ci < CA) {
                const int64_t idx =
                    UPA ? ((((int64_t)(zz >> 1) * Xh + (xx >> 1)) * Yh + (yy >> 1)) * CA + ci)
                        : ((((int64_t)zz * s.X + xx) * s.Y + yy) * CA + ci);
                piece[i] = *(const bf16x8*)(s.a + idx);
            } else {
                piece[i] = *(const bf16x8*)(s.b + (((int64_t)zz * s.X + xx) * s.Y + yy) * CB + (ci - CA));
            }
        }
    }
    // where the lane's 16 bytes of each chunk lie, relative to its voxel
    int off[KC];
#pragma unroll
    for (int i = 0; i < KC; ++i) {
        const int k = i * 32 + 8 * g;
        const int tap = k / CIN, ci = k - tap * CIN;
        off[i] = tap < kTaps ? ((tap / 9 * HX + tap / 3 % 3) * HY + tap % 3) * SV + ci : -1;
    }
    int vox[MTW];
#pragma unroll
    for (int t = 0; t < MTW; ++t) {
        const int v = (wm * MTW + t) * 16 + m;
        vox[t] = ((v / (BX * BY) * HX + v / BY % BX) * HY + v % BY) * SV;
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = tid + i * NTHR;
        if (e < PIECES) *(bf16x8*)(sm + e / PV * SV + 8 * (e % PV)) = piece[i];
    }
    if (tid == 0) *(bf16x8*)(sm + HV * SV) = bf16x8{};
    __syncthreads();
    f32x4 acc[MTW][NTW];
#pragma unroll
    for (int t = 0; t < MTW; ++t)
#pragma unroll
        for (int n = 0; n < NTW; ++n) acc[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    const bf16x8* wf = (const bf16x8*)w + lane;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
        bf16x8 A[NTW];
#pragma unroll
        for (int n = 0; n < NTW; ++n) A[n] = wf[(int64_t)((wn * NTW + n) * KC + kc) * 64];
#pragma unroll
        for (int t = 0; t < MTW; ++t) {
            // past the last tap: the zero piece
            const bf16x8 B = *(const bf16x8*)(sm + (off[kc] >= 0 ? vox[t] + off[kc] : HV * SV));
#pragma unroll
            for (int n = 0; n < NTW; ++n)
                acc[t][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[n], B, acc[t][n], 0, 0, 0);
        }
    }
    // the lane holds channels 16n + 4g .. + 3 of voxel 16t + m
#pragma unroll
    for (int t = 0; t < MTW; ++t) {
        const int v = (wm * MTW + t) * 16 + m;
        const int z = z0 + v / (BX * BY), x = x0 + v / BY % BX, y = y0 + v % BY;
        if (z >= s.Z || x >= s.X || y >= s.Y) continue;
        const int64_t gv = ((int64_t)z * s.X + x) * s.Y + y;
#pragma unroll
        for (int n = 0; n < NTW; ++n) {
            const int co = (wn * NTW + n) * 16 + 4 * g;
            if constexpr (MODE == MODE_RELU) {
                const f32x4 bias = *(const f32x4*)(o.bias + co);
                bf16x4 r;
#pragma unroll
                for (int j = 0; j < 4; ++j) r[j] = (bf16)fmaxf(acc[t][n][j] + bias[j], 0.f);
                *(bf16x4*)(o.o1 + gv * CO + co) = r;
            } else if constexpr (MODE == MODE_F32) {
                if (co == 0) o.of[gv] = acc[t][n][0] + o.bias[0];
            } else {
                bf16x4 r;
#pragma unroll
                for (int j = 0; j < 4; ++j) r[j] = (bf16)acc[t][n][j];
                if (co < o.split) {
                    if (o.mask) {
                        const bf16x4 y4 = *(const bf16x4*)(o.mask + gv * o.split + co);
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            if (!((float)y4[j] > 0.f)) r[j] = (bf16)0.f;
                    }
                    *(bf16x4*)(o.o1 + gv * o.split + co) = r;
                } else {
                    *(bf16x4*)(o.o2 + gv * (CO - o.split) + (co - o.split)) = r;
                }
            }
        }
    }
}

// Weight gradient dW[co][tap][ci] = sum_v G[v][co] X[v + tap][ci] and bias
// gradient sum_v G[v][co]: workgroup (x, y) sums the bricks x, x + gridDim.x, ...
// of 4 x 4 x 16 voxels for output channels [16 (y / NI), +16) and input channels
// [16 (y % NI), +16) of all 27 taps, and writes its sums to slice x of `part`.
//
// A brick's G and X (X with its halo) are staged once for all taps, transposed
// to [channel][voxel], as the matrix cores want eight consecutive voxels
// (reduction) of one channel per lane.  Along y a tap shifts the eight voxels by
// one, which would misalign the 16-byte reads, so X is kept in three copies, each
// shifted by one voxel; z and x shifts are whole rows.  Each wavefront takes
// 64 of the brick's voxels for all taps: 27 accumulator tiles.  The slices are
// added up by wgrad_sum_kernel in a fixed order.  One launch per tap restaging
// both operands with scalar LDS stores and adding to dW with atomics took
// 40-90 us a layer (48^3 network grid); this takes
// 11-24, all layers' sums together 16.
constexpr int kWgZ = 4, kWgX = 4, kWgY = 16;
constexpr int kWgRows = (kWgZ + 2) * (kWgX + 2);        // rows of 16 voxels of X
constexpr int kWgXs = kWgRows * kWgY + 8;               // one channel of one copy of X
constexpr int kWgGs = kWgZ * kWgX * kWgY + 8;           // one channel of G

template <int CA, int CB, bool UPA, int CO>
__global__ void __launch_bounds__(256) conv3_wgrad_kernel(ConvSrc s, const bf16* __restrict__ gy,
                                                          float* __restrict__ part, int64_t slice) {
    constexpr int CIN = CA + CB, NI = CIN / 16;
    static_assert(CA % 16 == 0 && CB % 16 == 0 && CO % 16 == 0, "channel blocking");
    __shared__ __attribute__((aligned(16))) bf16 Xt[3 * 16 * kWgXs];
    __shared__ __attribute__((aligned(16))) bf16 Gt[16 * kWgGs];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m = lane & 15, g = lane >> 4;
    const int c0 = blockIdx.y / NI * 16, i0 = blockIdx.y % NI * 16;
    const int by = (s.Y + kWgY - 1) / kWgY, bx = (s.X + kWgX - 1) / kWgX, bz = (s.Z + kWgZ - 1) / kWgZ;
    const int Xh = s.X >> 1, Yh = s.Y >> 1;
    f32x4 acc[kTaps];
#pragma unroll
    for (int t = 0; t < kTaps; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    float bsum[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) bsum[e] = 0.f;
    // eight channels [i0 + 8h, +8) of X at a voxel, zero outside the grid
    auto loadx = [&](int z, int x, int y, int h) {
        bf16x8 v = bf16x8{};
        if (z >= 0 && z < s.Z && x >= 0 && x < s.X && y >= 0 && y < s.Y) {
            const int ci = i0 + 8 * h;
            if (CB == 0 || ci < CA) {
                const int64_t idx = UPA ? ((((int64_t)(z >> 1) * Xh + (x >> 1)) * Yh + (y >> 1)) * CA + ci)
                                        : ((((int64_t)z * s.X + x) * s.Y + y) * CA + ci);
                v = *(const bf16x8*)(s.a + idx);
            } else {
                v = *(const bf16x8*)(s.b + (((int64_t)z * s.X + x) * s.Y + y) * CB + (ci - CA));
            }
        }
        return v;
    };
    for (int brick = blockIdx.x; brick < bz * bx * by; brick += gridDim.x) {
        const int y0 = brick % by * kWgY, x0 = brick / by % bx * kWgX, z0 = brick / (by * bx) * kWgZ;
        // X: unit u = voxel pair (two consecutive y of a row) and channel half
        constexpr int XU = kWgRows * (kWgY / 2) * 2;  // 576
#pragma unroll
        for (int i = 0; i < (XU + 255) / 256; ++i) {
            const int u = tid + i * 256;
            if (u < XU) {
                const int yp = u % 8, row = u / 8 % kWgRows, h = u / (8 * kWgRows);
                const int z = z0 + row / (kWgX + 2) - 1, x = x0 + row % (kWgX + 2) - 1, y = y0 + 2 * yp;
                bf16x8 v[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] = loadx(z, x, y - 1 + k, h);
                bf16* dst = Xt + 8 * h * kWgXs + row * kWgY + 2 * yp;
                // copy d holds voxel y + d - 1 at place y
#pragma unroll
                for (int d = 0; d < 3; ++d)
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        *(bf16x2*)(dst + (d * 16 + e) * kWgXs) = bf16x2{v[d][e], v[d + 1][e]};
            }
        }
        // G: 8 voxel pairs x 16 rows x 2 channel halves, one per thread
        {
            const int yp = tid % 8, row = tid / 8 % 16, h = tid / 128;
            const int z = z0 + row / kWgX, x = x0 + row % kWgX, y = y0 + 2 * yp;
            bf16x8 v[2];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                v[k] = bf16x8{};
                if (z < s.Z && x < s.X && y + k < s.Y)
                    v[k] = *(const bf16x8*)(gy + (((int64_t)z * s.X + x) * s.Y + y + k) * CO + c0 + 8 * h);
            }
            bf16* dst = Gt + 8 * h * kWgGs + row * kWgY + 2 * yp;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                *(bf16x2*)(dst + e * kWgGs) = bf16x2{v[0][e], v[1][e]};
                bsum[e] += (float)v[0][e] + (float)v[1][e];
            }
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            // chunk: 32 voxels, rows 4 wave + 2c and the next; lane's eight: row + g / 2, half g % 2
            const int r = 4 * wave + 2 * c + (g >> 1);
            const bf16x8 A = *(const bf16x8*)(Gt + m * kWgGs + r * kWgY + 8 * (g & 1));
            const int xr = (r / kWgX) * (kWgX + 2) + r % kWgX;  // the row at tap (0, 0)
            const bf16* xb = Xt + m * kWgXs + xr * kWgY + 8 * (g & 1);
#pragma unroll
            for (int t = 0; t < kTaps; ++t) {
                const bf16x8 B = *(const bf16x8*)(xb + (t % 3) * 16 * kWgXs +
                                                  (t / 9 * (kWgX + 2) + t / 3 % 3) * kWgY);
                acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A, B, acc[t], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // sum over the four wavefronts through LDS (27 x 64 x 16 bytes a wavefront), two rounds
    static_assert(sizeof(Xt) >= 2 * kTaps * 64 * sizeof(f32x4), "reduction fits the staging area");
    f32x4* red = (f32x4*)Xt;
#pragma unroll
    for (int half = 2; half >= 1; half >>= 1) {
        if (wave >= half && wave < 2 * half) {
#pragma unroll
            for (int t = 0; t < kTaps; ++t) red[((wave - half) * kTaps + t) * 64 + lane] = acc[t];
        }
        __syncthreads();
        if (wave < half) {
#pragma unroll
            for (int t = 0; t < kTaps; ++t) acc[t] += red[(wave * kTaps + t) * 64 + lane];
        }
        __syncthreads();
    }
    // D row 4g + j is output channel c0 + 4g + j, column m input channel i0 + m
    float* out = part + (int64_t)blockIdx.x * slice;
    if (wave == 0) {
#pragma unroll
        for (int t = 0; t < kTaps; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                out[((int64_t)(c0 + 4 * g + j) * kTaps + t) * CIN + i0 + m] = acc[t][j];
    }
    if (i0 == 0) {  // bias: sum the 128 threads of each channel half
        float* bs = (float*)Gt;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
#pragma unroll
            for (int q = 32; q > 0; q >>= 1) bsum[e] += __shfl_xor(bsum[e], q);
            if (lane == 0) bs[wave * 8 + e] = bsum[e];
        }
        __syncthreads();
        if (tid < 16) {
            const int h = tid / 8, e = tid % 8;
            out[(int64_t)CO * kTaps * CIN + c0 + tid] = bs[2 * h * 8 + e] + bs[(2 * h + 1) * 8 + e];
        }
    }
}

// grad = sum of a layer's slices: layer l's parameters (weights, then biases)
// are grad[first_l ..), its slices nslice_l of that length at part + at_l.
constexpr int kMaxLayers = 11;
struct WgradSum {
    int64_t first[kMaxLayers + 1];
    int64_t at[kMaxLayers];
    int nslice[kMaxLayers];
};
// 64 parameters a workgroup, each summed by four threads over a quarter of the slices.
__global__ void __launch_bounds__(256) wgrad_sum_kernel(float* __restrict__ grad,
                                                        const float* __restrict__ part, WgradSum a) {
    __shared__ float q[4][64];
    const int lane = threadIdx.x & 63, grp = threadIdx.x >> 6;
    const int64_t i = (int64_t)blockIdx.x * 64 + lane;
    float s = 0.f;
    if (i < a.first[kMaxLayers]) {
        int l = 0;
        while (i >= a.first[l + 1]) ++l;
        const int64_t n = a.first[l + 1] - a.first[l];
        const float* p = part + a.at[l] + (i - a.first[l]);
        const int per = (a.nslice[l] + 3) / 4, end = min(a.nslice[l], (grp + 1) * per);
#pragma unroll 8
        for (int k = grp * per; k < end; ++k) s += p[k * n];
    }
    q[grp][lane] = s;
    __syncthreads();
    if (grp == 0 && i < a.first[kMaxLayers]) grad[i] = (q[0][lane] + q[1][lane]) + (q[2][lane] + q[3][lane]);
}

// coarse[zc, xc, yc][c] = mean (or sum, zero where mask is not positive) of the
// 2x2x2 children; eight channels a thread.
template <bool MEAN>
__global__ void pool_kernel(bf16* __restrict__ out, const bf16* __restrict__ in,
                            const bf16* __restrict__ mask, int Zc, int Xc, int Yc, int C) {
    const int64_t n = (int64_t)Zc * Xc * Yc * (C / 8);
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int c = (int)(i % (C / 8)) * 8;
    int64_t r = i / (C / 8);
    const int yc = (int)(r % Yc);
    r /= Yc;
    const int xc = (int)(r % Xc), zc = (int)(r / Xc);
    const int X = 2 * Xc, Y = 2 * Yc;
    bf16x8 v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k)
        v[k] = *(const bf16x8*)(in + ((((int64_t)(2 * zc + (k >> 2)) * X + 2 * xc + (k >> 1 & 1)) * Y) +
                                      2 * yc + (k & 1)) * C + c);
    bf16x8 res;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) s += (float)v[k][e];
        res[e] = (bf16)(MEAN ? s * 0.125f : s);
    }
    if (!MEAN) {
        const bf16x8 y = *(const bf16x8*)(mask + 8 * i);
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (!((float)y[e] > 0.f)) res[e] = (bf16)0.f;
    }
    *(bf16x8*)(out + 8 * i) = res;
}

// fine[v][c] += coarse[parent(v)][c] / 8 (backward of the average pooling),
// zeroed where mask[v][c] is not positive; eight channels a thread.
__global__ void pool_back_kernel(bf16* __restrict__ fine, const bf16* __restrict__ coarse,
                                 const bf16* __restrict__ mask, int Z, int X, int Y, int C) {
    const int64_t n = (int64_t)Z * X * Y * (C / 8);
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int c = (int)(i % (C / 8)) * 8;
    int64_t r = i / (C / 8);
    const int y = (int)(r % Y);
    r /= Y;
    const int x = (int)(r % X), z = (int)(r / X);
    const int64_t p = ((((int64_t)(z >> 1) * (X >> 1) + (x >> 1)) * (Y >> 1)) + (y >> 1)) * C + c;
    bf16x8 f = *(const bf16x8*)(fine + 8 * i);
    const bf16x8 q = *(const bf16x8*)(coarse + p), act = *(const bf16x8*)(mask + 8 * i);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const bf16 t = (bf16)((float)f[e] + 0.125f * (float)q[e]);
        f[e] = (float)act[e] > 0.f ? t : (bf16)0.f;
    }
    *(bf16x8*)(fine + 8 * i) = f;
}

// FP64 partial sums.  DIFF = false: part[2b + 1] = sum a^2.  DIFF = true:
// e = a - b / (rms L^2) with rms from stats (sum f^2 over n), part[2b] = sum e,
// part[2b + 1] = sum e^2.
template <bool DIFF>
__global__ void sums_kernel(double* __restrict__ part, const float* __restrict__ a,
                            const float* __restrict__ b, const double* __restrict__ stats,
                            float len2, int64_t n) {
    double sc = 0.0;
    if (DIFF) {
        const double ms = stats[1] / (double)n;
        sc = ms > 0 ? 1.0 / (sqrt(ms) * (double)len2) : 0.0;
    }
    double s1 = 0.0, s2 = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        if (DIFF) {
            const double e = (double)a[i] - sc * (double)b[i];
            s1 += e;
            s2 += e * e;
        } else {
            const double e = a[i];
            s2 += e * e;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        s1 += __shfl_xor(s1, o);
        s2 += __shfl_xor(s2, o);
    }
    __shared__ double l1[4], l2[4];
    if ((threadIdx.x & 63) == 0) {
        l1[threadIdx.x >> 6] = s1;
        l2[threadIdx.x >> 6] = s2;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = l1[0] + l1[1] + l1[2] + l1[3];
        part[2 * blockIdx.x + 1] = l2[0] + l2[1] + l2[2] + l2[3];
    }
}

__global__ void sums_final_kernel(double* __restrict__ out, const double* __restrict__ part,
                                  int nparts) {
    double s1 = 0.0, s2 = 0.0;
    for (int i = threadIdx.x; i < nparts; i += blockDim.x) {
        s1 += part[2 * i];
        s2 += part[2 * i + 1];
    }
    for (int o = 32; o > 0; o >>= 1) {
        s1 += __shfl_xor(s1, o);
        s2 += __shfl_xor(s2, o);
    }
    __shared__ double l1[4], l2[4];
    if ((threadIdx.x & 63) == 0) {
        l1[threadIdx.x >> 6] = s1;
        l2[threadIdx.x >> 6] = s2;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        out[0] = l1[0] + l1[1] + l1[2] + l1[3];
        out[1] = l2[0] + l2[1] + l2[2] + l2[3];
    }
}

// Network input: channel 0 = f / rms(f), channel 1 = level set / L, others 0.
// stats[1] holds sum f^2 (from sums_kernel<false>).
__global__ void input_kernel(bf16* __restrict__ x, const float* __restrict__ f,
                             const float* __restrict__ ls, const double* __restrict__ stats,
                             float inv_len, int64_t V) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const double ms = stats[1] / (double)V;
    const float inv_rms = ms > 0 ? (float)(1.0 / sqrt(ms)) : 0.f;
    bf16x8 a = bf16x8{}, b = bf16x8{};
    a[0] = (bf16)(f[v] * inv_rms);
    a[1] = (bf16)(ls[v] * inv_len);
    *(bf16x8*)(x + v * kIn) = a;
    *(bf16x8*)(x + v * kIn + 8) = b;
}

// p0 = network output * rms(f) * L^2
__global__ void output_kernel(float* __restrict__ p, const float* __restrict__ out,
                              const double* __restrict__ stats, float len2, int64_t V) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const double ms = stats[1] / (double)V;
    p[v] = (float)((double)out[v] * sqrt(ms) * (double)len2);
}

// Loss gradient: target t = p / (rms(f) L^2); e = out - t; loss = mean
// (e - mean e)^2 (the pressure is defined up to a constant); g = 2 (e - e_bar) / V
// into channel 0 of a 16-channel BF16 gradient.  lsum[0] = sum e, lsum[1] = sum e^2.
__global__ void loss_grad_kernel(bf16* __restrict__ g, const float* __restrict__ out,
                                 const float* __restrict__ p, const double* __restrict__ stats,
                                 const double* __restrict__ lsum, float len2, float gscale,
                                 int64_t V) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const double ms = stats[1] / (double)V;
    const double sc = ms > 0 ? 1.0 / (sqrt(ms) * (double)len2) : 0.0;
    const double ebar = lsum[0] / (double)V;
    const double e = (double)out[v] - sc * (double)p[v];
    bf16x8 a = bf16x8{}, b = bf16x8{};
    a[0] = (bf16)((float)(2.0 * (e - ebar) / (double)V) * gscale);
    *(bf16x8*)(g + v * 16) = a;
    *(bf16x8*)(g + v * 16 + 8) = b;
}

// BF16 weights of every layer in the order conv3_kernel reads them: chunk kc of
// channel tile n is 64 lanes of eight values, lane 16 g + m holding row 16 n + m,
// k = 32 kc + 8 g + e.  Forward (wk): rows co, k = tap * CIN + ci; input gradient
// (wt): rows ci, k = (26 - tap) * CO + co.  k past the last tap stays zero.
struct PackLayers {
    int64_t first[kMaxLayers + 1];  // first parameter of layer l's weights
    bf16 *wk[kMaxLayers], *wt[kMaxLayers];
    int co[kMaxLayers], cin[kMaxLayers];
};
__device__ __forceinline__ int64_t frag_pos(int row, int k, int kp) {
    return ((((int64_t)(row >> 4) * (kp >> 5) + (k >> 5)) * 64) + ((k >> 3) & 3) * 16 + (row & 15)) * 8 + (k & 7);
}
__device__ __forceinline__ void pack_one(const PackLayers& a, int64_t i, float w) {
    int l = 0;
    while (i >= a.first[l + 1]) ++l;
    const int CO = a.co[l], CIN = a.cin[l];
    const int r = (int)(i - a.first[l]);
    if (r >= CO * kTaps * CIN) return;  // a bias
    const int ci = r % CIN, tap = r / CIN % kTaps, co = r / (CIN * kTaps);
    const bf16 v = (bf16)w;
    a.wk[l][frag_pos(co, tap * CIN + ci, kpad(CIN))] = v;
    a.wt[l][frag_pos(ci, (kTaps - 1 - tap) * CO + co, kpad(CO))] = v;
}
__global__ void pack_kernel(const float* __restrict__ w, PackLayers a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < a.first[kMaxLayers]) pack_one(a, i, w[i]);
}

// Adam (bias-corrected) over the flat parameter vector; grads are divided by
// gscale first (the loss gradient is scaled up to keep BF16 gradients normal).
// Writes the new weights' BF16 forms too.
__global__ void adam_kernel(float* __restrict__ w, float* __restrict__ m1, float* __restrict__ m2,
                            const float* __restrict__ grad, const uint8_t* __restrict__ frozen,
                            float lr, float b1, float b2, float eps, float c1, float c2,
                            float inv_gscale, PackLayers pk) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= pk.first[kMaxLayers] || frozen[i]) return;
    const float gi = grad[i] * inv_gscale;
    const float a = b1 * m1[i] + (1.f - b1) * gi;
    const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
    m1[i] = a;
    m2[i] = b;
    const float nw = w[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
    w[i] = nw;
    pack_one(pk, i, nw);
}

// Network grid from a finer one: the mean of each F^3 block of fine cells.
__global__ void down_kernel(float* __restrict__ out, const float* __restrict__ in, int Zc, int Xc,
                            int Yc, int F) {
    const int64_t n = (int64_t)Zc * Xc * Yc;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int yc = (int)(i % Yc);
    const int64_t r = i / Yc;
    const int xc = (int)(r % Xc), zc = (int)(r / Xc);
    const int64_t X = (int64_t)Xc * F, Y = (int64_t)Yc * F;
    float s = 0.f;
    for (int a = 0; a < F; ++a)
#pragma unroll 4
        for (int b = 0; b < F; ++b) {
            const float* row = in + (((int64_t)zc * F + a) * X + (int64_t)xc * F + b) * Y + (int64_t)yc * F;
#pragma unroll 4
            for (int d = 0; d < F; ++d) s += row[d];
        }
    out[i] = s / (float)(F * F * F);
}

// Fine cell values by trilinear interpolation of the network output at cell
// centres (coarse coordinate (i + 1/2) / F - 1/2, clamped at the walls), times
// rms(f) * L^2 * scale.
// A (64, 4) block over (y, x) and four z planes (the extents are multiples of 4):
// the FP64 scale, whose square root had cost more than the rest of a cell, is
// formed once per workgroup, the x and y weights once per column (192^3 from
// 48^3: 35 -> 19 us).  P2: F is a power of two, so 1 / F is exact and the coordinate a
// product; else it is divided (192^3 by 4 that way 21 us), since the reciprocal's
// rounding would move it and cells on coarse centres would mix two values.
constexpr int kUpZ = 4;
template <bool P2>
__global__ void __launch_bounds__(256) up_kernel(float* __restrict__ p, const float* __restrict__ out,
                                                 const double* __restrict__ stats, float len2, int Zc,
                                                 int Xc, int Yc, int F) {
    __shared__ double rms;
    if (threadIdx.x == 0 && threadIdx.y == 0)
        rms = sqrt(stats[1] / ((double)Zc * Xc * Yc));
    const int X = Xc * F, Y = Yc * F, Z = Zc * F;
    const int y = blockIdx.x * 64 + threadIdx.x, x = blockIdx.y * 4 + threadIdx.y;
    const float inv_f = 1.f / (float)F;
    auto axis = [&](int c, int nc, int& c0, int& c1, float& w) {
        const float v = (float)c + 0.5f;
        float u = (P2 ? v * inv_f : v / (float)F) - 0.5f;
        u = fminf(fmaxf(u, 0.f), (float)(nc - 1));
        c0 = (int)u;
        c1 = c0 + 1 < nc ? c0 + 1 : c0;
        w = u - (float)c0;
    };
    int x0, x1, y0, y1;
    float wx, wy;
    axis(min(x, X - 1), Xc, x0, x1, wx);
    axis(min(y, Y - 1), Yc, y0, y1, wy);
    float v[kUpZ];
#pragma unroll
    for (int k = 0; k < kUpZ; ++k) {
        int z0, z1;
        float wz;
        axis(blockIdx.z * kUpZ + k, Zc, z0, z1, wz);
        auto at = [&](int a, int b, int c) { return out[((int64_t)a * Xc + b) * Yc + c]; };
        const float v0 = (1.f - wx) * ((1.f - wy) * at(z0, x0, y0) + wy * at(z0, x0, y1)) +
                         wx * ((1.f - wy) * at(z0, x1, y0) + wy * at(z0, x1, y1));
        const float v1 = (1.f - wx) * ((1.f - wy) * at(z1, x0, y0) + wy * at(z1, x0, y1)) +
                         wx * ((1.f - wy) * at(z1, x1, y0) + wy * at(z1, x1, y1));
        v[k] = (1.f - wz) * v0 + wz * v1;
    }
    __syncthreads();
    const double r = rms;
    if (y >= Y || x >= X) return;
#pragma unroll
    for (int k = 0; k < kUpZ; ++k) {
        const int64_t z = (int64_t)blockIdx.z * kUpZ + k;
        if (z < Z) p[y + (int64_t)Y * (x + (int64_t)X * z)] = (float)((double)v[k] * r * (double)len2);
    }
}

}  // namespace unet
}  // namespace whhd

// ---------------------------------------------------------------------------
// Network and handle
// ---------------------------------------------------------------------------
namespace {
using whhd::unet::bf16;

// Layer table: (CA, CB, upsample a, CO, level).  CO of the last layer is 16
// with rows 1..15 held at zero.
struct LayerDef {
    int ca, cb;
    bool up;
    int co, level;
};
constexpr int kLayers = 11;
constexpr LayerDef kNet[kLayers] = {
    {16, 0, false, 16, 0},  // e0a = relu(conv(x))
    {16, 0, false, 16, 0},  // e0
    {16, 0, false, 32, 1},  // e1a = relu(conv(pool(e0)))
    {32, 0, false, 32, 1},  // e1
    {32, 0, false, 64, 2},  // ba = relu(conv(pool(e1)))
    {64, 0, false, 64, 2},  // b
    {64, 32, true, 32, 1},  // d1a = relu(conv([up(b), e1]))
    {32, 0, false, 32, 1},  // d1
    {32, 16, true, 16, 0},  // d0a = relu(conv([up(d1), e0]))
    {16, 0, false, 16, 0},  // d0
    {16, 0, false, 16, 0},  // out = conv(d0), channel 0
};
}  // namespace

struct whhd_unet_s {
    int nx, ny, nz;   // network grid
    int factor = 1;   // fine grid = factor * network grid
    float *fc = nullptr, *lsc = nullptr, *pc = nullptr;  // inputs averaged to the network grid
    int64_t V[3];
    int64_t woff[kLayers], boff[kLayers], nparams = 0;
    float *w = nullptr, *m1 = nullptr, *m2 = nullptr, *grad = nullptr;
    uint8_t* frozen = nullptr;
    bf16 *wk[kLayers] = {}, *wt[kLayers] = {};
    // activations
    bf16 *x = nullptr, *e0a = nullptr, *e0 = nullptr, *p0 = nullptr, *e1a = nullptr, *e1 = nullptr,
         *p1 = nullptr, *ba = nullptr, *b = nullptr, *d1a = nullptr, *d1 = nullptr, *d0a = nullptr,
         *d0 = nullptr;
    float* out = nullptr;
    // gradients
    bf16 *g0a = nullptr, *g0b = nullptr, *u0 = nullptr, *ge0 = nullptr, *g1a = nullptr,
         *g1b = nullptr, *u1 = nullptr, *ge1 = nullptr, *g1c = nullptr, *g2a = nullptr,
         *g2b = nullptr, *g2c = nullptr;
    float* wpart = nullptr;   // slices of the weight gradients (WgradSum)
    whhd::unet::WgradSum wsum;
    whhd::unet::PackLayers pack;
    double* part = nullptr;   // partial sums (2 * kParts) + stats[2] + lsum[2]
    double* host = nullptr;   // pinned copy of lsum
    int64_t step = 0;
    float gscale = 1.f;  // loss-gradient scale (divided out before Adam)
    double out_scale = 1.0;  // output units: p = output * rms(f) * L^2 * out_scale
    std::vector<void*> owned;
};

namespace whhd {
namespace unet {
namespace {

constexpr int kParts = 512;

#define TRY(e) do { int s_ = (e); if (s_ != WHHD_OK) return s_; } while (0)

int check_launch(const char* what) {
    set_last_kernel(what);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? WHHD_OK : hip_fail(e, what);
}

dim3 g1(int64_t n) { return dim3((unsigned)((n + 255) / 256)); }

template <int CA, int CB, bool UP, int CO, int MODE, int BZ, int BX, int BY, int WM, int WN>
void conv_launch(const ConvSrc& s, const bf16* w, const ConvOut& o, hipStream_t st) {
    const int64_t bricks = (int64_t)((s.Z + BZ - 1) / BZ) * ((s.X + BX - 1) / BX) * ((s.Y + BY - 1) / BY);
    hipLaunchKernelGGL((conv3_kernel<CA, CB, UP, CO, MODE, BZ, BX, BY, WM, WN>), dim3((unsigned)bricks),
                       dim3(64 * WM * WN), 0, st, s, w, o);
}

// Slices of layer l's weight gradient: workgroups for every CU (a slice has one
// per pair of channel blocks, two fit a CU), with the bricks spread evenly.
int wgrad_slices(int l, int Z, int X, int Y) {
    const int bricks = ((Z + kWgZ - 1) / kWgZ) * ((X + kWgX - 1) / kWgX) * ((Y + kWgY - 1) / kWgY);
    const int pairs = (kNet[l].ca + kNet[l].cb) / 16 * (kNet[l].co / 16);
    const int most = std::max(1, std::min(bricks, (pairs == 1 ? 256 : 512) / pairs));
    const int rounds = (bricks + most - 1) / most;
    return (bricks + rounds - 1) / rounds;
}

template <int CA, int CB, bool UP, int CO>
void wgrad_launch(whhd_unet_s* h, int l, const ConvSrc& s, const bf16* gy, hipStream_t st) {
    constexpr int CIN = CA + CB;
    hipLaunchKernelGGL((conv3_wgrad_kernel<CA, CB, UP, CO>),
                       dim3((unsigned)h->wsum.nslice[l], CIN / 16 * (CO / 16)), dim3(256), 0, st, s, gy,
                       h->wpart + h->wsum.at[l], (int64_t)CO * (kTaps * CIN + 1));
}

// forward of layer l (RELU into o1, or F32 for the last).  Bricks of 128 voxels
// on the finest level, 64 and 16 or 32 on the coarser ones, whose grids are small
// (64 -> 64 at 12^3, 2 x 2 x 4 voxels and four wavefronts 5.8 us, 2 x 4 x 4 and eight
// 7.0, and four 10.9); four to twelve wavefronts a brick.
int fwd_layer(whhd_unet_s* h, int l, const ConvSrc& s, bf16* out_bf, hipStream_t st) {
    ConvOut o{out_bf, nullptr, h->out, h->w + h->boff[l], nullptr, 0};
    const bf16* w = h->wk[l];
    switch (l) {
    case 0: case 1: case 9: conv_launch<16, 0, false, 16, MODE_RELU, 4, 4, 8, 4, 1>(s, w, o, st); break;
    case 2: conv_launch<16, 0, false, 32, MODE_RELU, 4, 4, 4, 4, 2>(s, w, o, st); break;
    case 3: case 7: conv_launch<32, 0, false, 32, MODE_RELU, 4, 4, 4, 4, 2>(s, w, o, st); break;
    case 4: conv_launch<32, 0, false, 64, MODE_RELU, 2, 2, 4, 1, 4>(s, w, o, st); break;
    case 5: conv_launch<64, 0, false, 64, MODE_RELU, 2, 2, 4, 1, 4>(s, w, o, st); break;
    case 6: conv_launch<64, 32, true, 32, MODE_RELU, 4, 4, 4, 4, 2>(s, w, o, st); break;
    case 8: conv_launch<32, 16, true, 16, MODE_RELU, 4, 4, 8, 4, 1>(s, w, o, st); break;
    default: conv_launch<16, 0, false, 16, MODE_F32, 4, 4, 8, 4, 1>(s, w, o, st); break;
    }
    return check_launch("unet_conv3_kernel");
}

// input gradient of layer l from its output gradient G (CO_l channels):
// channels [0, split) into o1, zero where mask is not positive, and [split, CIN)
// into o2
int bwd_data(whhd_unet_s* h, int l, const bf16* G, int Z, int X, int Y, bf16* o1, const bf16* mask,
             bf16* o2, int split, hipStream_t st) {
    const ConvSrc s{G, nullptr, Z, X, Y};
    const ConvOut o{o1, o2, nullptr, nullptr, mask, split};
    const bf16* w = h->wt[l];
    switch (l) {
    case 1: case 9: case 10: conv_launch<16, 0, false, 16, MODE_GRAD, 4, 4, 8, 4, 1>(s, w, o, st); break;
    case 2: conv_launch<32, 0, false, 16, MODE_GRAD, 4, 4, 4, 4, 1>(s, w, o, st); break;
    case 3: case 7: conv_launch<32, 0, false, 32, MODE_GRAD, 4, 4, 4, 4, 2>(s, w, o, st); break;
    case 4: conv_launch<64, 0, false, 32, MODE_GRAD, 2, 4, 4, 2, 2>(s, w, o, st); break;
    case 5: conv_launch<64, 0, false, 64, MODE_GRAD, 2, 2, 4, 1, 4>(s, w, o, st); break;
    case 6: conv_launch<32, 0, false, 96, MODE_GRAD, 4, 4, 4, 2, 6>(s, w, o, st); break;
    case 8: conv_launch<16, 0, false, 48, MODE_GRAD, 4, 4, 8, 4, 1>(s, w, o, st); break;
    default: return fail(WHHD_INVALID_ARG, "unet: no input gradient for the first layer");
    }
    return check_launch("unet_conv3_kernel(grad)");
}

int bwd_weight(whhd_unet_s* h, int l, const ConvSrc& s, const bf16* G, hipStream_t st) {
    switch (l) {
    case 0: case 1: case 9: case 10: wgrad_launch<16, 0, false, 16>(h, l, s, G, st); break;
    case 2: wgrad_launch<16, 0, false, 32>(h, l, s, G, st); break;
    case 3: case 7: wgrad_launch<32, 0, false, 32>(h, l, s, G, st); break;
    case 4: wgrad_launch<32, 0, false, 64>(h, l, s, G, st); break;
    case 5: wgrad_launch<64, 0, false, 64>(h, l, s, G, st); break;
    case 6: wgrad_launch<64, 32, true, 32>(h, l, s, G, st); break;
    default: wgrad_launch<32, 16, true, 16>(h, l, s, G, st); break;
    }
    return check_launch("unet_conv3_wgrad_kernel");
}

int pool(bf16* out, const bf16* in, const bf16* mask, int Zc, int Xc, int Yc, int C, bool mean,
         hipStream_t st) {
    const int64_t n = (int64_t)Zc * Xc * Yc * (C / 8);
    if (mean) hipLaunchKernelGGL(pool_kernel<true>, g1(n), dim3(256), 0, st, out, in, mask, Zc, Xc, Yc, C);
    else hipLaunchKernelGGL(pool_kernel<false>, g1(n), dim3(256), 0, st, out, in, mask, Zc, Xc, Yc, C);
    return check_launch("unet_pool_kernel");
}

int pool_back(bf16* fine, const bf16* coarse, const bf16* mask, int Z, int X, int Y, int C,
              hipStream_t st) {
    hipLaunchKernelGGL(pool_back_kernel, g1((int64_t)Z * X * Y * (C / 8)), dim3(256), 0, st, fine, coarse,
                       mask, Z, X, Y, C);
    return check_launch("unet_pool_back_kernel");
}

double* stats(whhd_unet_s* h) { return h->part + 2 * kParts; }
double* lsum(whhd_unet_s* h) { return h->part + 2 * kParts + 2; }

int forward(whhd_unet_s* h, const float* f, const float* ls, float len, hipStream_t st) {
    const int Z = h->nz, X = h->nx, Y = h->ny;
    const int64_t V0 = h->V[0];
    hipLaunchKernelGGL(sums_kernel<false>, dim3(kParts), dim3(256), 0, st, h->part, f, f,
                       (const double*)nullptr, 0.f, V0);
    hipLaunchKernelGGL(sums_final_kernel, dim3(1), dim3(256), 0, st, stats(h), h->part, kParts);
    hipLaunchKernelGGL(input_kernel, g1(V0), dim3(256), 0, st, h->x, f, ls, stats(h), 1.f / len, V0);
    TRY(check_launch("unet_input_kernel"));
    TRY(fwd_layer(h, 0, {h->x, nullptr, Z, X, Y}, h->e0a, st));
    TRY(fwd_layer(h, 1, {h->e0a, nullptr, Z, X, Y}, h->e0, st));
    TRY(pool(h->p0, h->e0, nullptr, Z / 2, X / 2, Y / 2, 16, true, st));
    TRY(fwd_layer(h, 2, {h->p0, nullptr, Z / 2, X / 2, Y / 2}, h->e1a, st));
    TRY(fwd_layer(h, 3, {h->e1a, nullptr, Z / 2, X / 2, Y / 2}, h->e1, st));
    TRY(pool(h->p1, h->e1, nullptr, Z / 4, X / 4, Y / 4, 32, true, st));
    TRY(fwd_layer(h, 4, {h->p1, nullptr, Z / 4, X / 4, Y / 4}, h->ba, st));
    TRY(fwd_layer(h, 5, {h->ba, nullptr, Z / 4, X / 4, Y / 4}, h->b, st));
    TRY(fwd_layer(h, 6, {h->b, h->e1, Z / 2, X / 2, Y / 2}, h->d1a, st));
    TRY(fwd_layer(h, 7, {h->d1a, nullptr, Z / 2, X / 2, Y / 2}, h->d1, st));
    TRY(fwd_layer(h, 8, {h->d1, h->e0, Z, X, Y}, h->d0a, st));
    TRY(fwd_layer(h, 9, {h->d0a, nullptr, Z, X, Y}, h->d0, st));
    return fwd_layer(h, 10, {h->d0, nullptr, Z, X, Y}, nullptr, st);
}

// loss = mean((e - e_bar)^2) into lsum (sum e, sum e^2), its gradient into
// h->grad
int backward(whhd_unet_s* h, const float* p, float len, hipStream_t st) {
    const int Z = h->nz, X = h->nx, Y = h->ny;
    const int Z1 = Z / 2, X1 = X / 2, Y1 = Y / 2, Z2 = Z / 4, X2 = X / 4, Y2 = Y / 4;
    const int64_t V0 = h->V[0], V1 = h->V[1], V2 = h->V[2];
    const float len2 = (float)((double)len * len * h->out_scale);
    hipLaunchKernelGGL(sums_kernel<true>, dim3(kParts), dim3(256), 0, st, h->part, h->out, p,
                       stats(h), len2, V0);
    hipLaunchKernelGGL(sums_final_kernel, dim3(1), dim3(256), 0, st, lsum(h), h->part, kParts);
    hipLaunchKernelGGL(loss_grad_kernel, g1(V0), dim3(256), 0, st, h->g0a, h->out, p, stats(h),
                       lsum(h), len2, h->gscale, V0);
    TRY(check_launch("unet_loss_kernels"));
    // out = conv(d0)
    TRY(bwd_weight(h, 10, {h->d0, nullptr, Z, X, Y}, h->g0a, st));
    TRY(bwd_data(h, 10, h->g0a, Z, X, Y, h->g0b, h->d0, nullptr, 16, st));
    // d0 = relu(conv(d0a))
    TRY(bwd_weight(h, 9, {h->d0a, nullptr, Z, X, Y}, h->g0b, st));
    TRY(bwd_data(h, 9, h->g0b, Z, X, Y, h->g0a, h->d0a, nullptr, 16, st));
    // d0a = relu(conv([up(d1), e0]))
    TRY(bwd_weight(h, 8, {h->d1, h->e0, Z, X, Y}, h->g0a, st));
    TRY(bwd_data(h, 8, h->g0a, Z, X, Y, h->u0, nullptr, h->ge0, 32, st));
    TRY(pool(h->g1a, h->u0, h->d1, Z1, X1, Y1, 32, false, st));  // up backward: sum of the children
    // d1 = relu(conv(d1a))
    TRY(bwd_weight(h, 7, {h->d1a, nullptr, Z1, X1, Y1}, h->g1a, st));
    TRY(bwd_data(h, 7, h->g1a, Z1, X1, Y1, h->g1b, h->d1a, nullptr, 32, st));
    // d1a = relu(conv([up(b), e1]))
    TRY(bwd_weight(h, 6, {h->b, h->e1, Z1, X1, Y1}, h->g1b, st));
    TRY(bwd_data(h, 6, h->g1b, Z1, X1, Y1, h->u1, nullptr, h->ge1, 64, st));
    TRY(pool(h->g2a, h->u1, h->b, Z2, X2, Y2, 64, false, st));
    // b = relu(conv(ba))
    TRY(bwd_weight(h, 5, {h->ba, nullptr, Z2, X2, Y2}, h->g2a, st));
    TRY(bwd_data(h, 5, h->g2a, Z2, X2, Y2, h->g2b, h->ba, nullptr, 64, st));
    // ba = relu(conv(pool(e1)))
    TRY(bwd_weight(h, 4, {h->p1, nullptr, Z2, X2, Y2}, h->g2b, st));
    TRY(bwd_data(h, 4, h->g2b, Z2, X2, Y2, h->g2c, nullptr, nullptr, 32, st));
    TRY(pool_back(h->ge1, h->g2c, h->e1, Z1, X1, Y1, 32, st));
    // e1 = relu(conv(e1a))
    TRY(bwd_weight(h, 3, {h->e1a, nullptr, Z1, X1, Y1}, h->ge1, st));
    TRY(bwd_data(h, 3, h->ge1, Z1, X1, Y1, h->g1a, h->e1a, nullptr, 32, st));
    // e1a = relu(conv(pool(e0)))
    TRY(bwd_weight(h, 2, {h->p0, nullptr, Z1, X1, Y1}, h->g1a, st));
    TRY(bwd_data(h, 2, h->g1a, Z1, X1, Y1, h->g1c, nullptr, nullptr, 16, st));
    TRY(pool_back(h->ge0, h->g1c, h->e0, Z, X, Y, 16, st));
    // e0 = relu(conv(e0a))
    TRY(bwd_weight(h, 1, {h->e0a, nullptr, Z, X, Y}, h->ge0, st));
    TRY(bwd_data(h, 1, h->ge0, Z, X, Y, h->g0b, h->e0a, nullptr, 16, st));
    // e0a = relu(conv(x))
    TRY(bwd_weight(h, 0, {h->x, nullptr, Z, X, Y}, h->g0b, st));
    hipLaunchKernelGGL(wgrad_sum_kernel, dim3((unsigned)((h->nparams + 63) / 64)), dim3(256), 0, st, h->grad,
                       h->wpart, h->wsum);
    return check_launch("unet_wgrad_sum_kernel");
}

// `in` on the network grid: itself, or its F^3 block means in `buf`.
const float* coarse(whhd_unet_s* h, float* buf, const float* in, hipStream_t st) {
    if (h->factor == 1) return in;
    hipLaunchKernelGGL(down_kernel, g1(h->V[0]), dim3(256), 0, st, buf, in, h->nz, h->nx, h->ny,
                       h->factor);
    return buf;
}

int pack_all(whhd_unet_s* h, hipStream_t st) {
    hipLaunchKernelGGL(pack_kernel, g1(h->nparams), dim3(256), 0, st, h->w, h->pack);
    return check_launch("unet_pack_kernel");
}

// deterministic He-normal initial weights (splitmix64 + Box-Muller), zero biases
void init_weights(std::vector<float>& w, const whhd_unet_s* h, uint64_t seed) {
    uint64_t st = seed;
    auto next = [&]() {
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    };
    auto unif = [&]() { return ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0); };
    w.assign(h->nparams, 0.f);
    for (int l = 0; l < kLayers; ++l) {
        const int cin = kNet[l].ca + kNet[l].cb;
        const int co_real = l == kLayers - 1 ? 1 : kNet[l].co;
        const int cin_real = l == 0 ? 2 : cin;
        const double sd = std::sqrt(2.0 / (kTaps * cin_real));
        for (int co = 0; co < co_real; ++co)
            for (int t = 0; t < kTaps; ++t)
                for (int ci = 0; ci < cin_real; ++ci) {
                    const double u1 = unif(), u2 = unif();
                    const double n = std::sqrt(-2.0 * std::log(u1)) * std::cos(6.283185307179586 * u2);
                    w[h->woff[l] + ((int64_t)co * kTaps + t) * cin + ci] = (float)(sd * n);
                }
    }
}

}  // namespace
}  // namespace unet
}  // namespace whhd

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
namespace {
void unet_release(whhd_unet_s* h) {
    if (!h) return;
    for (void* p : h->owned) (void)hipFree(p);
    if (h->host) (void)hipHostFree(h->host);
    delete h;
}
}  // namespace

extern "C" {

WHHD_API int whhd_unet_create(int nx, int ny, int nz, int factor, unsigned long long seed,
                              whhd_unet_t* out) {
    using namespace whhd;
    using namespace whhd::unet;
    if (!out) return fail(WHHD_INVALID_ARG, "unet_create: null handle pointer");
    *out = nullptr;
    if (factor < 1 || factor > 16) return fail(WHHD_INVALID_ARG, "unet_create: factor out of range");
    const int q = 4 * factor;
    if (nx < q || ny < q || nz < q || nx % q || ny % q || nz % q)
        return fail(WHHD_INVALID_ARG, "unet_create: extents must be multiples of 4 * factor");
    if ((int64_t)nx * ny * nz * 96 >= ((int64_t)1 << 40))
        return fail(WHHD_INVALID_ARG, "unet_create: grid too large");
    auto* h = new whhd_unet_s;
    h->factor = factor;
    nx /= factor;
    ny /= factor;
    nz /= factor;
    h->nx = nx; h->ny = ny; h->nz = nz;
    h->V[0] = (int64_t)nx * ny * nz;
    h->V[1] = h->V[0] / 8;
    h->V[2] = h->V[0] / 64;
    int64_t off = 0;
    for (int l = 0; l < kLayers; ++l) {
        const int cin = kNet[l].ca + kNet[l].cb;
        h->woff[l] = off;
        off += (int64_t)kNet[l].co * kTaps * cin;
        h->boff[l] = off;
        off += kNet[l].co;
    }
    h->nparams = off;
    bool ok = true;
    auto alloc = [&](size_t bytes) -> void* {
        void* p = nullptr;
        if (!ok || hipMalloc(&p, bytes) != hipSuccess) {
            ok = false;
            return nullptr;
        }
        h->owned.push_back(p);
        return p;
    };
    const size_t P = (size_t)h->nparams;
    h->w = (float*)alloc(P * 4);
    h->m1 = (float*)alloc(P * 4);
    h->m2 = (float*)alloc(P * 4);
    h->grad = (float*)alloc(P * 4);
    h->frozen = (uint8_t*)alloc(P);
    for (int l = 0; l < kLayers; ++l) {
        const int cin = kNet[l].ca + kNet[l].cb, co = kNet[l].co;
        h->wk[l] = (bf16*)alloc((size_t)co * kpad(cin) * 2);
        h->wt[l] = (bf16*)alloc((size_t)cin * kpad(co) * 2);
    }
    // slices of the weight gradients, layer after layer
    int64_t slices = 0;
    for (int l = 0; l < kLayers; ++l) {
        const int lv = kNet[l].level, cin = kNet[l].ca + kNet[l].cb;
        h->pack.first[l] = h->wsum.first[l] = h->woff[l];
        h->pack.wk[l] = h->wk[l];
        h->pack.wt[l] = h->wt[l];
        h->pack.co[l] = kNet[l].co;
        h->pack.cin[l] = cin;
        h->wsum.nslice[l] = wgrad_slices(l, nz >> lv, nx >> lv, ny >> lv);
        h->wsum.at[l] = slices;
        slices += h->wsum.nslice[l] * (int64_t)kNet[l].co * (kTaps * cin + 1);
    }
    h->pack.first[kLayers] = h->wsum.first[kLayers] = h->nparams;
    h->wpart = (float*)alloc((size_t)slices * 4);
    const int64_t V0 = h->V[0], V1 = h->V[1], V2 = h->V[2];
    auto act = [&](int64_t v, int c) { return (bf16*)alloc((size_t)v * c * 2); };
    h->x = act(V0, 16); h->e0a = act(V0, 16); h->e0 = act(V0, 16); h->p0 = act(V1, 16);
    h->e1a = act(V1, 32); h->e1 = act(V1, 32); h->p1 = act(V2, 32); h->ba = act(V2, 64);
    h->b = act(V2, 64); h->d1a = act(V1, 32); h->d1 = act(V1, 32); h->d0a = act(V0, 16);
    h->d0 = act(V0, 16);
    h->out = (float*)alloc((size_t)V0 * 4);
    h->g0a = act(V0, 16); h->g0b = act(V0, 16); h->u0 = act(V0, 32); h->ge0 = act(V0, 16);
    h->g1a = act(V1, 32); h->g1b = act(V1, 32); h->u1 = act(V1, 64); h->ge1 = act(V1, 32);
    h->g1c = act(V1, 16); h->g2a = act(V2, 64); h->g2b = act(V2, 64); h->g2c = act(V2, 32);
    h->part = (double*)alloc((2 * kParts + 4) * sizeof(double));
    if (factor > 1) {
        h->fc = (float*)alloc((size_t)V0 * 4);
        h->lsc = (float*)alloc((size_t)V0 * 4);
        h->pc = (float*)alloc((size_t)V0 * 4);
    }
    if (ok && hipHostMalloc((void**)&h->host, 4 * sizeof(double)) != hipSuccess) {
        h->host = nullptr;
        ok = false;
    }
    if (!ok) {
        unet_release(h);
        return fail(WHHD_OOM, "unet_create: allocation failed");
    }
    // zero everything the kernels do not always write (padded weight columns),
    // set the initial weights and the frozen mask (the last layer's rows 1..15)
    std::vector<float> w;
    init_weights(w, h, seed);
    std::vector<uint8_t> fr(P, 0);
    {
        const int l = kLayers - 1, cin = kNet[l].ca + kNet[l].cb;
        for (int co = 1; co < kNet[l].co; ++co) {
            for (int64_t k = 0; k < (int64_t)kTaps * cin; ++k) fr[h->woff[l] + co * kTaps * cin + k] = 1;
            fr[h->boff[l] + co] = 1;
        }
    }
    hipError_t e = hipSuccess;
    for (int l = 0; l < kLayers && e == hipSuccess; ++l) {
        const int cin = kNet[l].ca + kNet[l].cb, co = kNet[l].co;
        e = hipMemset(h->wk[l], 0, (size_t)co * kpad(cin) * 2);
        if (e == hipSuccess) e = hipMemset(h->wt[l], 0, (size_t)cin * kpad(co) * 2);
    }
    if (e == hipSuccess) e = hipMemcpy(h->w, w.data(), P * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(h->frozen, fr.data(), P, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(h->m1, 0, P * 4);
    if (e == hipSuccess) e = hipMemset(h->m2, 0, P * 4);
    if (e == hipSuccess) e = hipMemset(h->grad, 0, P * 4);
    if (e != hipSuccess) {
        unet_release(h);
        return hip_fail(e, "unet_create: initialisation");
    }
    int st = pack_all(h, nullptr);
    if (st == WHHD_OK && hipDeviceSynchronize() != hipSuccess) st = fail(WHHD_HIP_ERROR, "unet_create: sync");
    if (st != WHHD_OK) {
        unet_release(h);
        return st;
    }
    *out = h;
    return WHHD_OK;
}

WHHD_API long long whhd_unet_num_params(whhd_unet_t h) { return h ? h->nparams : -1; }

WHHD_API int whhd_unet_get_params(whhd_unet_t h, float* dst, int which) {
    using namespace whhd;
    if (!h || !dst) return fail(WHHD_INVALID_ARG, "unet_get_params: null argument");
    const float* src = which == 0 ? h->w : which == 1 ? h->grad : nullptr;
    if (!src) return fail(WHHD_INVALID_ARG, "unet_get_params: which is 0 (weights) or 1 (gradients)");
    hipError_t e = hipMemcpy(dst, src, (size_t)h->nparams * 4, hipMemcpyDeviceToHost);
    return e == hipSuccess ? WHHD_OK : hip_fail(e, "unet_get_params");
}

WHHD_API int whhd_unet_set_params(whhd_unet_t h, const float* src) {
    using namespace whhd;
    if (!h || !src) return fail(WHHD_INVALID_ARG, "unet_set_params: null argument");
    hipError_t e = hipMemcpy(h->w, src, (size_t)h->nparams * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemset(h->m1, 0, (size_t)h->nparams * 4);
    if (e == hipSuccess) e = hipMemset(h->m2, 0, (size_t)h->nparams * 4);
    if (e != hipSuccess) return hip_fail(e, "unet_set_params");
    h->step = 0;
    int st = unet::pack_all(h, nullptr);
    if (st == WHHD_OK && hipDeviceSynchronize() != hipSuccess)
        st = fail(WHHD_HIP_ERROR, "unet_set_params: sync");
    return st;
}

WHHD_API int whhd_unet_predict(whhd_unet_t h, float* p0, const float* f, const float* ls,
                               double length, void* stream) {
    using namespace whhd;
    if (!h || !p0 || !f || !ls || !(length > 0)) return fail(WHHD_INVALID_ARG, "unet_predict: bad argument");
    hipStream_t st = (hipStream_t)stream;
    const float* fin = unet::coarse(h, h->fc, f, st);
    const float* lin = unet::coarse(h, h->lsc, ls, st);
    int r = unet::forward(h, fin, lin, (float)length, st);
    if (r != WHHD_OK) return r;
    const float len2 = (float)(length * length * h->out_scale);
    if (h->factor == 1)
        hipLaunchKernelGGL(unet::output_kernel, unet::g1(h->V[0]), dim3(256), 0, st, p0, h->out,
                           unet::stats(h), len2, h->V[0]);
    else
        hipLaunchKernelGGL((h->factor & (h->factor - 1) ? unet::up_kernel<false> : unet::up_kernel<true>),
                           dim3((h->ny * h->factor + 63) / 64, (h->nx * h->factor + 3) / 4,
                                h->nz * h->factor / unet::kUpZ),
                           dim3(64, 4), 0, st, p0, h->out, unet::stats(h), len2, h->nz, h->nx, h->ny,
                           h->factor);
    return unet::check_launch("unet_output_kernel");
}

WHHD_API int whhd_unet_loss_grad(whhd_unet_t h, const float* f, const float* ls, const float* p,
                                 double length, double* loss, void* stream) {
    using namespace whhd;
    if (!h || !f || !ls || !p || !(length > 0)) return fail(WHHD_INVALID_ARG, "unet_loss_grad: bad argument");
    hipStream_t st = (hipStream_t)stream;
    const float* fin = unet::coarse(h, h->fc, f, st);
    const float* lin = unet::coarse(h, h->lsc, ls, st);
    const float* pin = unet::coarse(h, h->pc, p, st);
    int r = unet::forward(h, fin, lin, (float)length, st);
    if (r == WHHD_OK) r = unet::backward(h, pin, (float)length, st);
    if (r != WHHD_OK) return r;
    if (loss) {
        hipError_t e = hipMemcpyAsync(h->host, unet::lsum(h), 2 * sizeof(double),
                                      hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) return hip_fail(e, "unet_loss_grad: read-back");
        const double V = (double)h->V[0], m = h->host[0] / V;
        *loss = h->host[1] / V - m * m;
    }
    return WHHD_OK;
}

WHHD_API int whhd_unet_adam(whhd_unet_t h, float lr, void* stream) {
    using namespace whhd;
    if (!h || !(lr >= 0)) return fail(WHHD_INVALID_ARG, "unet_adam: bad argument");
    hipStream_t st = (hipStream_t)stream;
    const float b1 = 0.9f, b2 = 0.999f;
    h->step += 1;
    const float c1 = 1.f - std::pow(b1, (float)h->step), c2 = 1.f - std::pow(b2, (float)h->step);
    hipLaunchKernelGGL(unet::adam_kernel, unet::g1(h->nparams), dim3(256), 0, st, h->w, h->m1, h->m2,
                       h->grad, h->frozen, lr, b1, b2, 1e-8f, c1, c2, 1.f / h->gscale, h->pack);
    return unet::check_launch("unet_adam_kernel");
}

WHHD_API int whhd_unet_set_output_scale(whhd_unet_t h, double scale) {
    using namespace whhd;
    if (!h || !(scale > 0)) return fail(WHHD_INVALID_ARG, "unet_set_output_scale: bad argument");
    h->out_scale = scale;
    return WHHD_OK;
}

WHHD_API double whhd_unet_output_scale(whhd_unet_t h) { return h ? h->out_scale : 0.0; }

WHHD_API void whhd_unet_destroy(whhd_unet_t h) { unet_release(h); }

}  // extern "C"
