"""The DST solver's kernels at the lengths and line counts where they change: a line
per lane (FP32, 3..127 samples of 2^k - 1, and 255 from 8192 lines or 12288 contiguous
ones up; partial wavefronts, contiguous lines from buffers that are and are not
16-byte aligned), the half-wavefront transform below those counts, the folded sine
products (even and odd lengths around the strip widths and the largest folded length;
contiguous lines from memory up to 2^20 samples, staged in LDS above them) and the
tiled product beyond them (also for contiguous lines where neither pays).

Against dense FP64 sine transforms.  Tolerances: FP32 2e-5 relative, a few units
of roundoff per pass times the spread of the eigenvalues' reciprocals; FP64 1e-12.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3, 3), (7, 15, 1), (255, 5, 31), (63, 127, 9), (15, 255, 65), (31, 7, 127), (2, 5, 6),
          (16, 17, 33), (32, 31, 30), (97, 8, 64), (130, 129, 66), (4, 320, 5), (3, 321, 2), (257, 3, 5),
          (255, 91, 91), (111, 255, 111), (97, 85, 255),      # 255 samples, a line per lane
          (115, 96, 110), (81, 200, 160), (70, 201, 70), (40, 318, 101)]  # contiguous: LDS rows, tiled


def solve_dense(b, h):
    lam, t = [], b
    mats = []
    for d, hd in zip((0, 1, 2), (h[2], h[0], h[1])):
        n = b.shape[d]
        k = np.arange(1, n + 1)
        mats.append(np.sqrt(2.0 / (n + 1)) * np.sin(np.pi / (n + 1) * np.outer(k, k)))
        lam.append((2.0 * np.sin(np.pi * k / (2 * (n + 1))) / hd) ** 2)
    for inverse in (False, True):
        if inverse:
            t = t / (lam[0][:, None, None] + lam[1][None, :, None] + lam[2][None, None, :])
        for d, S in enumerate(mats):
            t = np.moveaxis(np.moveaxis(t, d, -1) @ S, -1, d)
    return t


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_dst_solve_lengths(whhd, shape, dtype):
    n1, n2, n3 = shape
    h = (0.02, 0.03, 0.025)
    rng = np.random.default_rng(n1 + 7 * n2 + 31 * n3)
    b = rng.standard_normal((n3, n1, n2)).astype(np.float32).astype(np.float64)
    ref = solve_dense(b, h)
    tol = 2e-5 if dtype == torch.float32 else 1e-12
    dst = whhd.CuDst3D(shape, h, dtype=dtype)
    for shift in (0, 1):      # elements past a 16-byte boundary
        src = torch.zeros(b.size + 4, dtype=dtype, device="cuda")[shift:shift + b.size]
        src.copy_(torch.from_numpy(b.reshape(-1)))
        out = torch.full((b.size + 4,), float("nan"), dtype=dtype, device="cuda")
        dst.Solve(out[shift:shift + b.size], src)
        torch.cuda.synchronize()
        got = out[shift:shift + b.size].cpu().numpy().astype(np.float64).reshape(b.shape)
        assert np.linalg.norm(got - ref) <= tol * np.linalg.norm(ref), shift
        assert torch.isnan(out[:shift]).all() and torch.isnan(out[shift + b.size:]).all()
        dst.Solve(src, src)   # in place
        torch.cuda.synchronize()
        assert np.array_equal(src.cpu().numpy().astype(np.float64).reshape(b.shape), got)
