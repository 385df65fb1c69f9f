"""The line-parallel kernels of every recovery pair (curl CDF3.7 / divergence
CDF4.6 and CDF3.5 / CDF4.4, either velocity bc, lines of 2^3..2^8 samples and
one more) and the launches that take a velocity's or potential's components
together.

Transforms: against the windowed kernels (the general path) on unconstrained
input, so that samples the boundary reflections ignore are covered too, and
against the FP64 oracle on admissible input.  Line counts of 64 k + r put
partial wavefronts at the end of the array.  A single array of few lines of 2^6
samples or more runs the windowed kernels by itself: the second test has the counts
from which such lines run the line-parallel ones, and the counts below.  Tolerances: FP32 roundoff over at
most eight lifting levels, 2e-6 relative to the FP64 oracle, hence twice that
between two FP32 paths.  Recovery: 1e-5 to the oracle, the path's stated bar.
"""
import numpy as np
import pytest
import torch

from _cases import bc_consistent, line_len
from waveletpotentials_amd import inputs as I

pytestmark = pytest.mark.gpu

PAIRS = [("cdf3.7", "cdf4.6"), ("cdf3.5", "cdf4.4")]
TOL32 = 2e-6
TOL_Q = 1e-5


def wtype(whhd, name):
    return whhd.WaveletType["WT_" + name.upper().replace(".", "_")]


def rel(a, b):
    a = np.concatenate([np.ravel(np.asarray(x, np.float64)) for x in a])
    b = np.concatenate([np.ravel(np.asarray(x, np.float64)) for x in b])
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def cuda(a):
    return torch.tensor(np.ascontiguousarray(a), dtype=torch.float32, device="cuda")


@pytest.mark.parametrize("wt", ["cdf3.7", "cdf4.6", "cdf3.5", "cdf4.4"])
@pytest.mark.parametrize("bc", ["n", "d"])
@pytest.mark.parametrize("axis", ["y", "x", "z"])
def test_line_parallel_equals_windowed(whhd, orc, wt, bc, axis):
    rng = np.random.default_rng(17)
    fw = whhd.CuWHHDForward.GetInstance()
    L = whhd.lib()
    for levels in (3, 4, 5, 6, 7, 8):
        n = line_len(wt, levels)
        for m1, m2 in ((1, 1), (37, 3), (64, 2)):
            shape = {"y": (m2, m1, n), "x": (m2, n, m1), "z": (n, m1, m2)}[axis]
            nz, nx, ny = shape
            free = rng.standard_normal(shape)
            good = np.moveaxis(bc_consistent(np.moveaxis(free, {"y": 2, "x": 1, "z": 0}[axis], -1),
                                             wt, bc), -1, {"y": 2, "x": 1, "z": 0}[axis])
            for x in (free, np.ascontiguousarray(good)):
                for fwd in (True, False):
                    got = []
                    for mode in (0, 1):
                        assert L.whhd_set_line_kernel(mode) == 0
                        try:
                            dst = torch.full(shape, float("nan"), device="cuda")
                            fw.Solve1D(dst, cuda(x), (nx, ny, nz), levels, axis, bc,
                                       wtype(whhd, wt), fwd)
                            torch.cuda.synchronize()
                        finally:
                            L.whhd_set_line_kernel(0)
                        got.append(dst.cpu().numpy())
                    assert rel([got[0]], [got[1]]) < 2 * TOL32, (n, m1, m2, fwd)
            ref, _ = orc.transform(np.ascontiguousarray(good), levels, axis, bc, wt, False)
            assert rel([got[0]], [ref]) < TOL32, (n, m1, m2)


@pytest.mark.parametrize("wt", ["cdf3.7", "cdf4.6", "cdf3.5", "cdf4.4"])
@pytest.mark.parametrize("bc", ["n", "d"])
@pytest.mark.parametrize("axis", ["y", "x", "z"])
def test_few_and_many_long_lines(whhd, wt, bc, axis):
    """Lines of 2^6..2^8 samples: up to 2048 of them (4096 contiguous ones, and x lines
    with fewer than 16 neighbours in memory) one line per wavefront, the windowed
    kernels' bits; more of them a line per lane, the same to FP32 rounding."""
    rng = np.random.default_rng(23)
    fw = whhd.CuWHHDForward.GetInstance()
    L = whhd.lib()
    for levels in (6, 7, 8):
        n = line_len(wt, levels)
        for m1, m2 in ((1, 1), (64, 32), (1, 2048), (683, 3), (65, 63), (8, 512), (8, 513), (241, 17)):
            shape = {"y": (m2, m1, n), "x": (m2, n, m1), "z": (n, m1, m2)}[axis]
            few = m1 * m2 <= (4096 if axis == "y" or (axis == "x" and m1 < 16) else 2048)
            nz, nx, ny = shape
            x = cuda(rng.standard_normal(shape))
            for fwd in (True, False):
                got = []
                for mode in (0, 1):
                    assert L.whhd_set_line_kernel(mode) == 0
                    try:
                        dst = torch.full(shape, float("nan"), device="cuda")
                        fw.Solve1D(dst, x, (nx, ny, nz), levels, axis, bc, wtype(whhd, wt), fwd)
                        torch.cuda.synchronize()
                    finally:
                        L.whhd_set_line_kernel(0)
                    got.append(dst.cpu().numpy())
                assert rel([got[0]], [got[1]]) < 2 * TOL32, (n, m1, m2, fwd)
                if few:
                    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32)), (n, m1, m2, fwd)


@pytest.mark.parametrize("pair", PAIRS, ids=["37-46", "35-44"])
@pytest.mark.parametrize("bc", ["n", "d"])
@pytest.mark.parametrize("n", [(8, 8, 8), (16, 8, 32), (4, 16, 8), (32, 64, 8), (64, 64, 64)])
def test_recover3d_pairs_match_oracle(whhd, orc, pair, bc, n):
    """Both forms of Solve; (4, 16, 8) has an x axis below the line-parallel kernels'
    range, so that grid is solved out of place, array by array."""
    nx, ny, nz = n
    dx = tuple(1.0 / v for v in n)
    rng = np.random.default_rng(nx + ny)
    q = [rng.standard_normal(s) for s in ((nz + 1, nx, ny + 1), (nz + 1, nx + 1, ny),
                                          (nz, nx + 1, ny + 1))]
    if bc == "n":
        q[0][[0, -1]] = 0; q[0][:, :, [0, -1]] = 0
        q[1][[0, -1]] = 0; q[1][:, [0, -1]] = 0
        q[2][:, [0, -1]] = 0; q[2][:, :, [0, -1]] = 0
    v = I.curl3d(*q, dx)
    ref = orc.recover3d(*v, n, dx, bc=bc, wt_curl=pair[0], wt_div=pair[1], with_vout=True)
    rec = whhd.CuWaveletPotentialRecover3D(n, dx, bc, wtype(whhd, pair[0]), wtype(whhd, pair[1]))
    out = [torch.full(r.shape, float("nan"), device="cuda") for r in ref]
    rec.Solve(*out, *(cuda(a) for a in v))
    torch.cuda.synchronize()
    got = [t.cpu().numpy() for t in out]
    assert all(np.isfinite(g).all() for g in got)
    assert rel(got[:3], ref[:3]) < TOL_Q
    assert rel(got[3:], ref[3:]) < TOL_Q
    out2 = [torch.full(r.shape, float("nan"), device="cuda") for r in ref[:3]]
    rec.Solve(*out2, *(cuda(a) for a in v))
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(out[:3], out2))


def test_traced_solve_equals_merged(whhd):
    """A traced solve runs the components one by one; the results are the same bits."""
    n = (64, 32, 64)
    nx, ny, nz = n
    T = whhd.WaveletType
    g = torch.Generator(device="cpu").manual_seed(3)
    v = [torch.randn(s, generator=g).cuda() for s in ((nz, nx + 1, ny), (nz, nx, ny + 1),
                                                      (nz + 1, nx, ny))]
    rec = whhd.CuWaveletPotentialRecover3D(n, tuple(1.0 / k for k in n), "n", T.WT_CDF3_7, T.WT_CDF4_6)
    a = [torch.full(s, float("nan"), device="cuda") for s in ((nz + 1, nx, ny + 1),
                                                              (nz + 1, nx + 1, ny), (nz, nx + 1, ny + 1))]
    b = [t.clone() for t in a]
    rec.Solve(*a, *v)
    rec.TraceBegin(1)
    rec.Solve(*b, *v)
    stages, solves = rec.TraceEnd()
    assert solves == 1 and len(stages) == 19
    assert all(torch.equal(x, y) for x, y in zip(a, b))
