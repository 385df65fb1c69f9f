"""The eikonal relaxation's skipping of tiles that cannot change: bit for bit the
relaxations of every tile, whatever the count.

A call of few relaxations runs every tile, so a long run must equal the same number
of relaxations taken seven at a time.  Tiles are 64 y x 4 x x 4 or 8 z, eight on
grids of at least 2048 of those, and one or two planes deep on grids that are: extents
around them with remainders, axes of one cell, values beyond the 1e8 that stands for the outside, infinities and NaN; and an
array of 2^31 bytes and more, whose offsets are 64-bit, against a narrow copy of it
whose are not.  The eight-plane tiles are held against the FP64 oracle too, at the
2e-6 of the solid-geometry tests.
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
                               (20, 50, 1), (70, 321, 150), (129, 130, 170),
                               (1030, 1020, 1), (730, 720, 2)])
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


def test_eight_plane_tiles_match_oracle(whhd, orc):
    n = (70, 321, 150)     # 6 x 18 x 19 = 2052 tiles
    nx, ny, nz = n
    h = 1.0 / max(n)
    z, x, y = np.meshgrid(*(np.arange(k) + 0.5 for k in (nz, nx, ny)), indexing="ij")
    d = np.sqrt((x - nx * 0.4) ** 2 + (y - ny * 0.6) ** 2 + (z - nz * 0.3) ** 2) * h - 0.05
    ls = np.where(d > 2 * h, 4.0, d).astype(np.float32)
    a = torch.from_numpy(ls).cuda()
    relax(whhd, a, n, h, 12)
    torch.cuda.synchronize()
    assert np.abs(a.cpu().numpy() - orc.eikonal_sweep(ls.astype(np.float64), h, 12)).max() < 2e-6


def test_64_bit_offsets(whhd):
    """820^3 cells (2.2 GB): a field constant along x, whose relaxation is that of
    eight of its columns.  826 relaxations leave tiles out, seven at a time do not."""
    n = 820
    h = 1.0 / n
    c = (torch.arange(n, device="cuda", dtype=torch.float64) + 0.5) * h
    d = (torch.sqrt((c[None, :] - 0.4) ** 2 + (c[:, None] - 0.6) ** 2) - 0.2).float()
    d = torch.where(d > 2 * h, torch.full_like(d, 4.0), d)
    narrow = d[:, None, :].expand(n, 8, n).contiguous()
    wide = d[:, None, :].expand(n, n, n).contiguous()
    for _ in range(118):
        relax(whhd, narrow, (8, n, n), h, 7)
    relax(whhd, wide, (n, n, n), h, 826)
    torch.cuda.synchronize()
    for k in range(0, n, 20):
        assert torch.equal(wide[k:k + 20].view(torch.int32), narrow[k:k + 20, :1].view(torch.int32).expand(20, n, n)), k


def test_long_run_beside_a_capture(whhd):
    """A run that leaves tiles out takes memory from its stream's pool: on a stream of
    its own while another one is being captured, and in a captured stream itself,
    where every tile runs.  The capture stays valid and all results agree."""
    n = (40, 70, 30)
    h = 1.0 / 70
    g = torch.Generator(device="cpu").manual_seed(4)
    ls = torch.rand((30, 40, 70), generator=g).cuda() - 0.2
    want = ls.clone()
    for _ in range(16):
        relax(whhd, want, n, h, 7)
    beside, inside, x = ls.clone(), ls.clone(), torch.ones(1000, device="cuda")
    scratch = [torch.empty_like(ls), torch.empty_like(ls)]
    other = torch.cuda.Stream()
    torch.cuda.synchronize()

    def run(t, k, stream):
        assert whhd.lib().whhd_eikonal_sweep(t.data_ptr(), scratch[k].data_ptr(), *n, ctypes.c_double(h), 112,
                                             ctypes.c_void_p(stream.cuda_stream)) == 0

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        x.mul_(2.0)
        run(beside, 0, other)
        run(inside, 1, torch.cuda.current_stream())
    torch.cuda.synchronize()
    assert torch.equal(beside, want)
    for k in range(3):
        inside.copy_(ls)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(inside, want)
        assert float(x[0]) == 2.0 ** (k + 1)
