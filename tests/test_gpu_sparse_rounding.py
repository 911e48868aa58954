"""Rounding of the sparse operator in crowded cells (work items, the terms of a
pool summed before they join the row): rows of several hundred to two thousand
terms against sums in extended precision, beside the same kernel values added
up one after another in index order.

Bar: no further off the extended sums than 1.25 times that plain sum (the
kernel values of both are within a few ulp; the bar leaves room for the
device's square root and for the sample of rows).
"""
import numpy as np
import pytest
import torch

import aboria_amd as ab

pytestmark = pytest.mark.gpu


def wendland(dx, r, kind):
    q = np.sqrt((dx.astype(kind) ** 2).sum(-1)) / kind(r)
    t = np.maximum(1 - q, 0)
    return t ** 4 * (4 * q + 1)


@pytest.mark.parametrize("dim,leaf,r", [(2, 4_000.0, 0.2), (3, 2_500.0, 0.3)])
def test_crowded_rows(ctx, dim, leaf, r):
    n = 20_011
    rng = np.random.default_rng(dim)
    low, high, per = [0.0] * dim, [1.0] * dim, [False] * dim
    cl = ab.CellListOrdered(ctx, low, high, per, leaf)
    cl.update_positions(torch.tensor(rng.random((n, dim)), device="cuda"))
    q = cl.positions().cpu().numpy()
    x = rng.random(n) + 0.5
    op = ab.SparseOperator(ctx, cl, cl.positions(), r, ab.Kernel.wendland_c2(r))
    y = op.apply_colmajor(torch.tensor(x[None].copy(), device="cuda"),
                          torch.zeros(1, n, dtype=torch.float64, device="cuda")).cpu().numpy()[0]
    rows = rng.choice(n, 400, replace=False)
    gpu, plain = 0.0, 0.0
    for i in rows:
        dx = q - q[i]
        j = np.flatnonzero((dx * dx).sum(-1) <= r * r)
        assert len(j) > 200  # (corner points have an eighth of a ball)
        exact = (wendland(dx[j], r, np.longdouble) * x[j].astype(np.longdouble)).sum()
        one = np.add.accumulate(wendland(dx[j], r, np.float64) * x[j])[-1]
        gpu += float((np.longdouble(y[i]) - exact) / exact) ** 2
        plain += float((np.longdouble(one) - exact) / exact) ** 2
    print("relative rounding: operator %.2e, one running sum %.2e"
          % (np.sqrt(gpu / len(rows)), np.sqrt(plain / len(rows))), flush=True)
    assert np.sqrt(gpu) <= 1.25 * np.sqrt(plain)
