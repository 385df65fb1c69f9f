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
