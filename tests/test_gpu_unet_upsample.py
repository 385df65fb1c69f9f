"""The prediction on a grid finer than the network's: block means in, trilinear
interpolation of the network's output back, for factors that are and are not
powers of two.

Against the FP64 oracle at 1e-2, the bar of test_gpu_unet.py.  At the cells that
lie on coarse centres (odd factors) the interpolation weights are exactly 0, so the
fine value is the network's own output: the same weights on the coarse grid give it
up to the rounding of the final scale, one unit in the last place (2^-23).  A
coordinate that is one rounding off gives weights of up to 2^-17 there (row 102 of
these grids) and misses that bound.
"""
import numpy as np
import pytest
import torch

from test_gpu_unet import effective, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("net_dims,factor", [((4, 8, 4), 3), ((8, 4, 12), 4), ((4, 4, 8), 6)])
def test_prediction_matches_oracle(whhd, orc, net_dims, factor):
    n = tuple(factor * v for v in net_dims)
    nx, ny, nz = n
    net = whhd.UNet3D(n, seed=2, factor=factor)
    rng = np.random.default_rng(factor)
    f = rng.standard_normal((nz, nx, ny)).astype(np.float32)
    ls = rng.uniform(-0.1, 0.4, (nz, nx, ny)).astype(np.float32)
    p0 = torch.full((nz, nx, ny), float("nan"), device="cuda")
    net.predict(p0, torch.from_numpy(f).cuda(), torch.from_numpy(ls).cuda(), 1.0)
    torch.cuda.synchronize()
    ref = orc.unet_predict(effective(orc, net.get_params()), f.astype(np.float64), ls.astype(np.float64), 1.0,
                           bf16=True, factor=factor)
    assert rel(p0.cpu().numpy(), ref) < 1e-2


@pytest.mark.parametrize("factor", [3, 5, 7, 9, 11, 13, 15])
def test_cells_on_coarse_centres_are_the_network_output(whhd, factor):
    net_dims = (4, 104, 4)
    nx, ny, nz = net_dims
    rng = np.random.default_rng(1)
    # eighths, constant over the blocks: every block mean is exact
    f = (rng.integers(-32, 33, (nz, nx, ny)) / 8).astype(np.float32)
    ls = (rng.integers(-8, 9, (nz, nx, ny)) / 8).astype(np.float32)
    fine = lambda a: np.kron(a, np.ones((factor,) * 3, np.float32))  # noqa: E731
    coarse_net = whhd.UNet3D(net_dims, seed=6)
    net = whhd.UNet3D(tuple(factor * v for v in net_dims), seed=6, factor=factor)
    want = torch.full((nz, nx, ny), float("nan"), device="cuda")
    got = torch.full(tuple(factor * v for v in (nz, nx, ny)), float("nan"), device="cuda")
    coarse_net.predict(want, torch.from_numpy(f).cuda(), torch.from_numpy(ls).cuda(), 1.0)
    net.predict(got, torch.from_numpy(fine(f)).cuda(), torch.from_numpy(fine(ls)).cuda(), 1.0)
    torch.cuda.synchronize()
    want = want.cpu().numpy()
    mid = slice(factor // 2, None, factor)
    got = got.cpu().numpy()[mid, mid, mid]
    assert np.isfinite(got).all()
    assert (np.abs(got - want) <= np.abs(want) * 2.0 ** -23).all()
