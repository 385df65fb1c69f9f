"""The U-Net's convolution and weight-gradient kernels on grids that do not fill
their bricks (4 x 4 x 8 voxels on the finest level, 4 x 4 x 4 and 2 x 4 x 4 below,
4 x 4 x 16 in the weight gradient): the smallest grid (one voxel on the coarsest
level), extents below a brick's and ragged ones, and a grid with several bricks
per weight-gradient slice.

Against the FP64 oracle rounding to BF16 where the GPU does, as
test_gpu_unet.py: prediction 1e-2, loss 1e-2, gradients 6e-2 per layer; twice
that below 4096 voxels, where a single ReLU or rounding flip weighs more.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(np.ravel(a) - np.ravel(b)) / max(np.linalg.norm(np.ravel(b)), 1e-300))


@pytest.mark.parametrize("dims", [(4, 4, 4), (20, 36, 4), (24, 12, 28), (8, 4, 68), (32, 40, 28)])
def test_network_on_ragged_grids_matches_oracle(whhd, orc, dims):
    nx, ny, nz = dims
    tol = 1.0 if nx * ny * nz >= 4096 else 2.0
    net = whhd.UNet3D(dims, seed=3)
    rng = np.random.default_rng(nx + ny)
    f = rng.standard_normal((nz, nx, ny)).astype(np.float32)
    ls = rng.uniform(-0.1, 0.4, (nz, nx, ny)).astype(np.float32)
    p = (rng.standard_normal((nz, nx, ny)) * 1e-2).astype(np.float32)
    d = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    w = net.get_params().astype(np.float64)
    lay, _ = orc.unet_layout()
    for wo, bo in lay:
        w[wo:bo] = orc.bf16_round(w[wo:bo])
    F, L, P = (a.astype(np.float64) for a in (f, ls, p))
    p0 = torch.full((nz, nx, ny), float("nan"), device="cuda")
    net.predict(p0, d(f), d(ls), 1.0)
    torch.cuda.synchronize()
    assert rel(p0.cpu().numpy(), orc.unet_predict(w, F, L, 1.0, bf16=True)) < tol * 1e-2
    loss = net.loss_grad(d(f), d(ls), d(p), 1.0)
    g = net.get_params(1).astype(np.float64)
    rloss, rg, _ = orc.unet_loss_grad(w, F, L, P, 1.0, bf16=True)
    assert abs(loss - rloss) <= tol * 1e-2 * rloss
    for l, (wo, bo) in enumerate(lay):
        co = orc.UNET_LAYERS[l][3]
        assert rel(g[wo:bo], rg[wo:bo]) < tol * 6e-2, f"layer {l} weights"
        if l < len(lay) - 1:
            assert rel(g[bo:bo + co], rg[bo:bo + co]) < tol * 6e-2, f"layer {l} biases"
    # the same inputs give the same bits (no atomics)
    assert net.loss_grad(d(f), d(ls), d(p), 1.0) == loss
    assert np.array_equal(net.get_params(1).astype(np.float64), g)
