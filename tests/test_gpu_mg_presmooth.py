"""The first two pre-smoothing sweeps of a level that starts from zero, in one pass.

Levels that are launched one by one (more than 4096 cells) with odd and even
extents, every wall condition, and one to five sweeps (one: the plain first sweep;
odd counts: the result has to end in the level's own array).  Plain V-cycles are
held against the FP64 oracle's at the tolerance of the V-cycle tests, 1e-4 relative
L2 after one and two cycles (FP32 rounding of the sweeps); conjugate gradients,
whose preconditioner starts the finest level from zero, have to reach their
tolerance in the oracle's FP64 residual (the V-cycle iteration by itself diverges on
this right-hand side).
"""
import numpy as np
import pytest
import torch

from test_gpu_mg import cuda, problem, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nu1", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n,bc", [((38, 44, 70), "n"), ((51, 34, 66), "d"), ((33, 130, 36), "z")])
def test_vcycles_match_oracle(whhd, orc, n, bc, nu1):
    fr, f, h = problem(orc, n, 11 + nu1)
    mg = whhd.CuMultigridFrac3D(*(cuda(a) for a in fr), n, h, bc)
    df = cuda(f)
    out = torch.empty_like(df)
    for k in (1, 2):
        mg.Solve(out, None, df, k, nu1, 2, 0.8)
        torch.cuda.synchronize()
        got = out.cpu().numpy().astype(np.float64)
        ref = orc.mg_solve(f.astype(np.float32).astype(np.float64), *fr, h, bc, n_iters=k, nu1=nu1, nu2=2,
                           weight=0.8)
        if bc == "n":
            got, ref = got - got.mean(), ref - ref.mean()
        assert rel(got, ref) < 1e-4


@pytest.mark.parametrize("nu", [1, 2, 3])
@pytest.mark.parametrize("n,bc", [((38, 44, 70), "n"), ((51, 34, 66), "d")])
def test_pcg_reaches_tolerance(whhd, orc, n, bc, nu):
    fr, f, h = problem(orc, n, 5)
    mg = whhd.CuMultigridFrac3D(*(cuda(a) for a in fr), n, h, bc)
    df = cuda(f)
    hi, lo = torch.empty_like(df), torch.empty_like(df)
    _, r, ok = mg.SolvePCG(hi, lo, None, df, 1e-6, 400, nu, nu)
    assert ok and r <= 1e-6
    v = hi.double().cpu().numpy() + lo.double().cpu().numpy()
    r_ref = orc.mg_rel_residual(v, f.astype(np.float32).astype(np.float64), *fr, h, bc)
    assert r_ref <= 1e-6 * (1 + 1e-3) + 1e-7


def test_create_allocates_what_a_solve_reads(whhd):
    """The device memory of a 192^3 handle: per level three cell arrays, the faces, and
    the reciprocal diagonals of the levels that are launched one by one (the finest in
    its FP16 form only); on the finest level FP16 faces and three more cell arrays.
    12 MB on top for the allocations' granularity and the small tables; one unread
    cell array of the finest level is 28 MB."""
    n = 192
    fr = [torch.ones(s, device="cuda") for s in ((n, n + 1, n), (n, n, n + 1), (n + 1, n, n))]
    h = (1.0 / n,) * 3
    del_first = whhd.CuMultigridFrac3D(*fr, (n, n, n), h, "n")   # the runtime's own first-use memory
    del del_first
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    mg = whhd.CuMultigridFrac3D(*fr, (n, n, n), h, "n")
    used = before - torch.cuda.mem_get_info()[0]
    want = 0
    for l, (x, y, z) in enumerate(mg.levels()):
        cells, faces = x * y * z, (x + 1) * y * z + x * (y + 1) * z + x * y * (z + 1)
        want += 4 * (3 * cells + faces) + (4 * 4 * cells + 2 * faces if l == 0 else 4 * cells)
    assert used <= want + (12 << 20), (used, want)
