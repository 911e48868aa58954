"""The batched dense operator in its symmetric form: problems below, at and
above the 1,024-row tile and its 256- and 64-column steps, among enough others
that the form is used, against the one-sided form (a set tile shape).

Bar: both sum the same kernel values, n terms per row in another order:
(n + 64) eps sum_j |K_ij x_j| in FP64, 2e-6 of it in FP32-compensated.
"""
import numpy as np
import pytest
import torch

import aboria_amd as ab

pytestmark = pytest.mark.gpu

KERNELS = {"multiquadric": ab.Kernel.multiquadric(0.05), "gaussian": ab.Kernel.gaussian(0.3),
           "inverse": ab.Kernel.smooth_inv_r(0.01)}


@pytest.mark.parametrize("name,dim", [("multiquadric", 2), ("gaussian", 3), ("inverse", 1),
                                      ("multiquadric", 3)])
def test_symmetric_matches_one_sided(ctx, name, dim):
    edges = [1, 63, 64, 1_023, 1_024, 1_025, 1_087, 1_088, 1_280, 1_281, 2_048, 2_049, 5_000]
    sizes = edges + [4_100] * 420  # 2,100 tiles of 1,024 rows and more
    off = np.concatenate([[0], np.cumsum(sizes)])
    n = int(off[-1])
    g = torch.Generator(device="cuda").manual_seed(dim)
    pos = torch.rand(n, dim, generator=g, device="cuda", dtype=torch.float64)
    x = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) - 0.5
    op = ab.DenseBatchOperator(ctx, off, pos, KERNELS[name])
    one = ab.DenseBatchOperator(ctx, off, pos, KERNELS[name])
    one.tune(ab.FP64, force=1)
    one.tune(ab.FP32_COMPENSATED, force=1)
    scale = one.apply(x.abs(), torch.zeros_like(x))
    rows = torch.tensor(np.repeat(sizes, sizes), device="cuda", dtype=torch.float64)
    ref = one.apply(x, torch.zeros_like(x))
    y = op.apply(x, torch.zeros_like(x))
    assert torch.all((y - ref).abs() <= (rows + 64) * 2.0 ** -52 * scale)
    assert not torch.equal(y, ref)  # the other form did run
    assert torch.equal(op.apply(x, torch.zeros_like(x)), y)  # the same bits again
    if name == "multiquadric":  # no further off the double-double sums
        exact = -op.residual_dd(torch.zeros_like(x), x)
        assert (y - exact).norm() <= 1.02 * (ref - exact).norm()
    # nothing was timed on the way: the tuner reports the symmetric form, whose
    # shape passed back keeps it and restores it after another was set
    rpt, ms = op.tune(ab.FP64)
    assert rpt == 4 and ms[4] > 0 and ms[1] == 0 and ms[2] == 0
    assert torch.equal(op.apply(x, torch.zeros_like(x)), y)
    one.tune(ab.FP64, force=rpt)
    assert torch.equal(one.apply(x, torch.zeros_like(x)), y)
    y32 = op.apply(x, torch.full_like(x, 0.25), ab.FP32_COMPENSATED) - 0.25
    assert torch.all((y32 - ref).abs() <= 2e-6 * scale + 2.0 ** -52)
