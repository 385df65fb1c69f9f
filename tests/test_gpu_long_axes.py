"""3D recovery by in-place passes where they are launched in another way than on a
small cube: every wavelet pair and velocity bc with one axis of 2^7 or 2^8 cells per
direction, y lines outside the line-parallel kernels' lengths (4 and 512 cells: the
windowed kernels on that axis, in place), and a grid above the size up to which the
three components share a launch.

Tolerances: 1e-5 relative to the FP64 oracle on the same FP32 input, the path's stated
bar, or four times the error of the oracle's own FP32 build where that is more (the
curl of white noise amplifies rounding by an amount that depends on the extents).
"""
import ctypes

import numpy as np
import pytest
import torch

from test_gpu_line_pairs import PAIRS, TOL_Q, cuda, rel, wtype
from waveletpotentials_amd import inputs as I

pytestmark = pytest.mark.gpu


def fp32_oracle(orc, v, n, dx, bc, pair):
    f, i = ctypes.c_float, ctypes.c_int
    P = ctypes.POINTER(f)
    fn = orc.lib_f32().orc_recover3d
    fn.argtypes = [P] * 9 + [i, i, i, f, f, f, ctypes.c_char, i, i]
    nx, ny, nz = n
    out = [np.zeros(s, np.float32) for s in ((nz + 1, nx, ny + 1), (nz + 1, nx + 1, ny), (nz, nx + 1, ny + 1))]
    out += [np.zeros_like(a) for a in v]
    p = lambda a: a.ctypes.data_as(P)  # noqa: E731
    assert fn(*(p(a) for a in out), *(p(a) for a in v), nx, ny, nz, *dx, bc.encode(), pair[0], pair[1]) == 0
    return out


def velocity(n, dx, bc, seed):
    """FP32 curl of a white-noise edge potential (no wall flux for bc 'n')."""
    nx, ny, nz = n
    rng = np.random.default_rng(seed)
    q = [rng.standard_normal(s) for s in ((nz + 1, nx, ny + 1), (nz + 1, nx + 1, ny), (nz, nx + 1, ny + 1))]
    if bc == "n":
        q[0][[0, -1]] = 0; q[0][:, :, [0, -1]] = 0
        q[1][[0, -1]] = 0; q[1][:, [0, -1]] = 0
        q[2][:, [0, -1]] = 0; q[2][:, :, [0, -1]] = 0
    return [np.ascontiguousarray(a, dtype=np.float32) for a in I.curl3d(*q, dx)]


@pytest.mark.parametrize("pair", PAIRS, ids=["37-46", "35-44"])
@pytest.mark.parametrize("bc", ["n", "d"])
@pytest.mark.parametrize("n", [(256, 8, 16), (16, 8, 256), (128, 256, 8), (8, 128, 16), (8, 4, 16), (16, 512, 8)])
def test_recovery_matches_oracle(whhd, orc, n, bc, pair):
    dx = tuple(1.0 / k for k in n)
    v = velocity(n, dx, bc, sum(n))
    ref = orc.recover3d(*(a.astype(np.float64) for a in v), n, dx, bc=bc, wt_curl=pair[0], wt_div=pair[1],
                        with_vout=True)
    wts = [wtype(whhd, w) for w in pair]
    low = fp32_oracle(orc, v, n, dx, bc, [int(w) for w in wts])
    rec = whhd.CuWaveletPotentialRecover3D(n, dx, bc, *wts)
    out = [torch.full(r.shape, float("nan"), device="cuda") for r in ref]
    rec.Solve(*out, *(cuda(a) for a in v))
    torch.cuda.synchronize()
    got = [t.cpu().numpy() for t in out]
    assert all(np.isfinite(g).all() for g in got)
    for part in (slice(0, 3), slice(3, 6)):
        tol = max(TOL_Q, 4 * rel(low[part], ref[part]))
        assert rel(got[part], ref[part]) < tol, tol
    out2 = [torch.full(r.shape, float("nan"), device="cuda") for r in ref[:3]]
    rec.Solve(*out2, *(cuda(a) for a in v))
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(out[:3], out2))


@pytest.mark.parametrize("bc", ["n", "d"])
def test_components_one_by_one_above_the_merged_size(whhd, bc):
    """256 x 512 x 256 (134 MB a component): a smooth potential, whose velocity the
    recovered one reproduces to the 1e-5 bar, and the windowed kernels' result."""
    n = (256, 512, 256)
    nx, ny, nz = n
    dx = tuple(1.0 / k for k in n)
    T = whhd.WaveletType

    def wave(k, count, centre):
        t = (torch.arange(count, device="cuda", dtype=torch.float64) + (0.5 if centre else 0.0)) / (
            count if centre else count - 1)
        return torch.cos(np.pi * k * t) if centre else torch.sin(np.pi * k * t)

    def comp(shape, own, k):
        z, x, y = (wave(k + d, c, d == own) for d, c in enumerate(shape))
        return z[:, None, None] * x[None, :, None] * y[None, None, :]

    q = [comp((nz + 1, nx, ny + 1), 1, 2), comp((nz + 1, nx + 1, ny), 2, 3), comp((nz, nx + 1, ny + 1), 0, 4)]

    def curl(a, b, c):
        hx, hy, hz = dx
        return [(c[:, :, 1:] - c[:, :, :-1]) / hy - (b[1:] - b[:-1]) / hz,
                (a[1:] - a[:-1]) / hz - (c[:, 1:, :] - c[:, :-1, :]) / hx,
                (b[:, 1:, :] - b[:, :-1, :]) / hx - (a[:, :, 1:] - a[:, :, :-1]) / hy]

    v = [t.contiguous() for t in curl(*q)]
    norm = lambda ts: float(sum(t.double().square().sum() for t in ts)) ** 0.5  # noqa: E731
    v32 = [t.float() for t in v]
    got = []
    for mode in (0, 1):
        assert whhd.lib().whhd_set_line_kernel(mode) == 0
        try:
            rec = whhd.CuWaveletPotentialRecover3D(n, dx, bc, T.WT_CDF3_7, T.WT_CDF4_6)
            out = [torch.full_like(t, float("nan"), dtype=torch.float32) for t in q]
            rec.Solve(*out, *v32)
            torch.cuda.synchronize()
        finally:
            whhd.lib().whhd_set_line_kernel(0)
        got.append(out)
    assert norm([a.double() - b.double() for a, b in zip(*got)]) < 2 * TOL_Q * norm(got[1])
    w = curl(*(t.double() for t in got[0]))
    assert norm([a - b for a, b in zip(w, v)]) < TOL_Q * norm(v)
