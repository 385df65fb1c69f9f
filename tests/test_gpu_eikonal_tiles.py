"""The eikonal relaxation's skipping of tiles that cannot change: bit for bit the
relaxations of every tile, whatever the count.

A call of fewer than eight relaxations runs every tile, so a long run must equal
the same number of relaxations taken seven at a time.  Extents around the tile
(64 y x 4 x x 16 z) with remainders, axes of one cell, values beyond the 1e8 that
stands for the outside, infinities and NaN.
"""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def relax(whhd, ls, n, h, iters):
    scratch = torch.full_like(ls, float("nan"))
    st = whhd.lib().whhd_eikonal_sweep(ls.data_ptr(), scratch.data_ptr(), *n, ctypes.c_double(h),
                                       iters, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == 0


@pytest.mark.parametrize("n", [(8, 64, 32), (9, 65, 33), (70, 130, 50), (1, 40, 20), (30, 1, 40),
                               (20, 50, 1)])
@pytest.mark.parametrize("special", [False, True])
def test_skipped_tiles_equal_every_tile(whhd, n, special):
    nx, ny, nz = n
    h = 1.0 / max(n)
    z, x, y = np.meshgrid(*(np.arange(k) + 0.5 for k in (nz, nx, ny)), indexing="ij")
    d = np.sqrt((x - nx * 0.4) ** 2 + (y - ny * 0.6) ** 2 + (z - nz * 0.3) ** 2) * h - 0.1
    ls = np.where(d > 2 * h, 4.0, d).astype(np.float32)
    if special:
        rng = np.random.default_rng(5)
        flat = ls.reshape(-1)
        at = rng.choice(flat.size, 40, replace=False)
        flat[at[:10]] = np.inf
        flat[at[10:20]] = 3e8
        flat[at[20:30]] = -2e8
        flat[at[30:]] = np.nan
    a, b = torch.from_numpy(ls).cuda(), torch.from_numpy(ls.copy()).cuda()
    total = 7 * max(8, 2 * max(n) // 7)
    relax(whhd, a, n, h, total)
    for _ in range(total // 7):
        relax(whhd, b, n, h, 7)
    torch.cuda.synchronize()
    assert np.array_equal(a.cpu().numpy().view(np.uint32), b.cpu().numpy().view(np.uint32))
