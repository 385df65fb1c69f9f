// Dispatch of the line-parallel kernels (line_parallel.h).  They are
// instantiated per recovery pair -- curl CDF3.7 or CDF3.5 on 2^L samples with
// divergence CDF4.6 or CDF4.4 on 2^L + 1, the curl wavelet with the velocity's
// bc 'n' or 'd' and the divergence wavelet with the other -- for L = 3..8, in
// lp_cdf*_*.hip.  A kernel holds both wavelets of its pair, so one launch can
// transform the three components of a velocity or potential along one axis.
#include <hip/hip_runtime.h>

#include <cstdio>

#include "line_parallel.h"
#include "whhd_internal.h"

namespace whhd {

#define WHHD_LP_PAIR(C, D)                                                                        \
    extern template bool lp_launch<C, D, true>(int, int, lp::LpJobs&, int, int, hipStream_t);  \
    extern template bool lp_launch<C, D, false>(int, int, lp::LpJobs&, int, int, hipStream_t);
WHHD_LP_PAIR(W_Cdf37N, W_Cdf46D)
WHHD_LP_PAIR(W_Cdf37D, W_Cdf46N)
WHHD_LP_PAIR(W_Cdf35N, W_Cdf44D)
WHHD_LP_PAIR(W_Cdf35D, W_Cdf44N)
#undef WHHD_LP_PAIR

// The instantiated pair a (wavelet, bc) belongs to (0..3, -1: none) and which
// of its two kinds it is (0: curl on 2^L samples, 1: divergence on 2^L + 1).
static int lp_pair(int wt, char bc, int* kind) {
    if (bc != 'n' && bc != 'd') return -1;
    switch (wt) {
    case WT_CDF3_7: *kind = 0; return bc == 'n' ? 0 : 1;
    case WT_CDF4_6: *kind = 1; return bc == 'd' ? 0 : 1;
    case WT_CDF3_5: *kind = 0; return bc == 'n' ? 2 : 3;
    case WT_CDF4_4: *kind = 1; return bc == 'd' ? 2 : 3;
    default: return -1;
    }
}

// Whether the interleaved passes of a pair exist along an axis of `levels`.
bool lp_interleaves(int wt_curl, char bc_curl, int wt_div, char bc_div, int levels) {
    int kc = 0, kd = 0;
    const int p = lp_pair(wt_curl, bc_curl, &kc);
    return p >= 0 && p == lp_pair(wt_div, bc_div, &kd) && kc == 0 && kd == 1 && levels >= 3 && levels <= 8;
}

// Returns WHHD_OK when a line-parallel kernel was launched, -1 when none fits
// (the caller then uses the tile kernel).  dst may equal src where a line is
// read ahead of its stores: the inverse, and either direction interleaved.
int lp_transform(const LineJob* jobs, int njobs, int levels, char axis, bool fwd, bool interleaved,
                 hipStream_t stream, int waves, int nb) {
    if (njobs < 1 || njobs > lp::kMaxJobs || levels < 3 || levels > 8) return -1;
    lp::LpJobs a{};
    a.n = njobs;
    int pair = -1;
    const bool contig = (axis == 'y' || axis == 'Y');
    for (int k = 0; k < njobs; ++k) {
        const LineJob& jb = jobs[k];
        if (jb.dst == jb.src && !jb.in_place) return -1;
        if (interleaved && contig) return -1;
        lp::LpGeom& g = a.j[k].g;
        g.batch_stride = jb.stride;
        int n;
        const int64_t nx = jb.nx, ny = jb.ny, nz = jb.nz;
        int64_t lines, inner, outer_stride, step;
        switch (axis) {
        case 'y': case 'Y':
            n = jb.ny; lines = nx * nz; inner = lines; outer_stride = 0; step = 1; break;
        case 'x': case 'X':
            n = jb.nx; lines = ny * nz; inner = ny; outer_stride = nx * ny; step = ny; break;
        case 'z': case 'Z':
            n = jb.nz; lines = ny * nx; inner = ny; outer_stride = ny; step = nx * ny; break;
        default: return -1;
        }
        // buffer offsets are 32-bit; keep clear of the out-of-range marker
        if (nx * ny * nz * 4 >= (int64_t)lp::kOutOfRange) return -1;
        g.total_lines = (uint32_t)lines;
        g.total_elems = (uint32_t)(nx * ny * nz);
        g.lines_inner = (uint32_t)inner;
        g.inner_stride = contig ? (uint32_t)ny : 1u;
        g.outer_stride = (uint32_t)outer_stride;
        g.step = (uint32_t)step;
        int kind = 0;
        const int p = lp_pair(jb.wt, jb.bc, &kind);
        if (p < 0 || (k > 0 && p != pair) || n != (1 << levels) + kind) return -1;
        pair = p;
        a.j[k].kind = kind;
        a.j[k].dst = jb.dst;
        a.j[k].src = jb.src;
    }
    bool ok = false;
    const int layout = contig ? lp::kContig : interleaved ? lp::kInterleaved : lp::kStrided;
#define WHHD_LP_RUN(C, D)                                                                  \
    ok = fwd ? lp_launch<C, D, true>(levels, layout, a, waves, nb, stream)                 \
             : lp_launch<C, D, false>(levels, layout, a, waves, nb, stream)
    switch (pair) {
    case 0: WHHD_LP_RUN(W_Cdf37N, W_Cdf46D); break;
    case 1: WHHD_LP_RUN(W_Cdf37D, W_Cdf46N); break;
    case 2: WHHD_LP_RUN(W_Cdf35N, W_Cdf44D); break;
    case 3: WHHD_LP_RUN(W_Cdf35D, W_Cdf44N); break;
    }
#undef WHHD_LP_RUN
    if (!ok) return -1;
    char name[96];
    std::snprintf(name, sizeof(name), "lp_kernel<%s %c,L=%d,%s,%s>", wavelet_name(jobs[0].wt), jobs[0].bc,
                  levels, fwd ? "fwd" : "inv", contig ? "contiguous" : "strided");
    set_last_kernel(name);
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? WHHD_OK : hip_fail(e, "line-parallel kernel");
}

}  // namespace whhd
