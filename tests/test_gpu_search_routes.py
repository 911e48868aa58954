"""Searches and operators at the sizes where the kernel that serves a query
changes: sets just below and above 16,384, cells of few and of many particles,
both at once, stencils of up to and beyond 125 buckets, periodic grids too
small for one bucket per stencil cell, centres other than the particles.

Bar: neighbour lists equal the oracle's as multisets per row and ascend within
a row where no bucket is visited twice; counts, the one-pass search and the
assembled operator give the same lists; FP64 operator within 1e-13 *
sum_j |f_ij x_j| of the oracle, FP32-compensated within 2e-6 of it.
"""
import numpy as np
import pytest
import torch

import aboria_amd as ab
import oracle

pytestmark = pytest.mark.gpu


def cloud(kind, n, dim, rng):
    if kind == "uniform":
        return rng.random((n, dim))
    # a fifth of the particles in one small blob, the rest spread out: cells of
    # every occupancy side by side
    k = n // 5
    blob = (0.0 if kind == "corner" else 0.3) + 0.02 * rng.standard_normal((k, dim))
    return np.concatenate([blob % 1.0, rng.random((n - k, dim))])


CASES = [
    # (kind, n, dim, periodic, n_leaf, radius in cells, other centres)
    ("uniform", 16_384, 3, False, 5.0, 1.0, 0),
    ("uniform", 16_385, 3, True, 5.0, 1.0, 0),
    ("uniform", 17_001, 3, False, 70.0, 0.95, 0),
    ("uniform", 17_001, 2, True, 90.0, 0.9, 0),
    ("blob", 20_003, 3, True, 2.0, 0.9, 0),
    ("blob", 20_003, 2, False, 3.0, 1.9, 0),
    ("blob", 17_003, 1, True, 6.0, 2.5, 0),
    ("uniform", 17_003, 3, False, 1.5, 2.5, 0),   # 343 buckets: work items only
    ("blob", 9_001, 3, False, 1.5, 2.4, 0),
    ("uniform", 40, 3, True, 10.0, 1.2, 0),       # 1 or 2 cells a side: images meet
    ("uniform", 17_000, 2, True, 9_000.0, 0.01, 0),
    ("blob", 20_003, 3, True, 4.0, 0.9, 17_111),
    ("blob", 20_003, 3, False, 4.0, 0.9, 333),
    ("uniform", 300, 2, False, 5.0, 1.0, 17_111),
]


# Runs of 100 to 160 and of 64 to 70 queries: their last few.
CASES += [
    ("uniform", 17_003, 2, False, 130.0, 0.5, 0),
    ("uniform", 17_003, 3, True, 65.0, 0.6, 0),
]


# Cells of few particles beside crowded ones, at domain faces too.
CASES += [
    ("blob", 17_003, 2, True, 10.0, 0.9, 0),
    ("blob", 30_001, 3, False, 6.0, 0.95, 0),
    ("blob", 20_003, 1, False, 8.0, 0.7, 0),
    ("corner", 20_003, 3, True, 5.0, 0.9, 0),
    ("corner", 20_003, 2, False, 5.0, 1.7, 0),
]
# Many centres: few tests in all, centres that share cells or do not, a radius
# well below a cell's side; most particles of a set of 12,300 in one bucket.
CASES += [
    ("uniform", 300, 2, False, 5.0, 1.0, 40_001),
    ("uniform", 8_000, 2, True, 900.0, 0.3, 33_003),   # 1,500 centres a cell
    ("uniform", 8_000, 2, False, 900.0, 0.3, 33_003),
    ("uniform", 16_000, 3, True, 60.0, 0.6, 17_111),
    ("uniform", 60_000, 2, False, 9.0, 0.95, 130_001),  # 20 to 30 centres a cell
    ("uniform", 300, 1, False, 3.0, 1.0, 1_000_003),
    ("uniform", 12_300, 2, False, 1e6, 0.1, 0),
]


@pytest.mark.parametrize("case", CASES, ids=["%s-%d-%dd-%s-%g-%g-%d" % c for c in CASES])
def test_routes(ctx, case):
    kind, n, dim, per, n_leaf, cells_r, other = case
    print("case", case, flush=True)
    rng = np.random.default_rng(n * 7 + dim)
    pos = cloud(kind, n, dim, rng)
    low, high, periodic = [0.0] * dim, [1.0] * dim, [per] * dim
    cl = ab.CellListOrdered(ctx, low, high, periodic, n_leaf)
    cl.update_positions(torch.tensor(pos, device="cuda"))
    oc = oracle.Cells(low, high, periodic, n_leaf)
    oc.update(pos.copy(), np.ones(n, np.uint8))
    r = cells_r / oc.grid[0]
    if other:
        centres = rng.uniform(-0.1, 1.1, (other, dim))
        centres[5, 0] = np.nan
        centres = torch.tensor(centres, device="cuda")
    else:
        centres = cl.positions()
    rp_o, col_o = oc.search(centres.cpu().numpy(), r)
    res = ab.euclidean_search(cl, centres, r)
    rp, col = res.row_ptr.cpu().numpy(), res.col.cpu().numpy()
    assert np.array_equal(rp, rp_o)
    row = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    assert np.array_equal(col[np.lexsort((col, row))], col_o[np.lexsort((col_o, row))])
    if oc.grid[0] > 6:
        same = row[1:] == row[:-1]
        assert np.all(col[1:][same] > col[:-1][same])
    search = ab.Search(cl, centres, r)
    one = torch.full((len(col) + 7,), -1, dtype=torch.int32, device="cuda")
    assert search.run_fused(cl, centres, r, one) == len(col)
    assert np.array_equal(one.cpu().numpy()[:len(col)], col)
    assert torch.all(one[len(col):] == -1)

    m = centres.shape[0]
    x = rng.standard_normal((n, 9))
    xt = torch.tensor(x.T.copy(), device="cuda")
    # (exp(-4 d^2 / r^2): in FP32 the rounding of d^2 and of the exponent adds up
    # to 1.5e-6 of a term at the cutoff)
    kern = (1, 0.5 * r)
    y_o = oc.sparse_matvec(centres.cpu().numpy(), r, kern, x)
    scale = oc.sparse_matvec(centres.cpu().numpy(), r, kern, np.abs(x))
    op = ab.SparseOperator(ctx, cl, centres, r, ab.Kernel.gaussian(0.5 * r))
    assert op.nnz == len(col)
    for precision, tol in ((ab.FP64, 1e-13), (ab.FP32_COMPENSATED, 2e-6)):
        for nrhs in (1, 2, 3, 5, 8, 9):
            y = torch.full((nrhs, m), 0.5, dtype=torch.float64, device="cuda")
            op.apply_colmajor(xt[:nrhs], y, precision)
            err = np.abs(y.cpu().numpy().T - 0.5 - y_o[:, :nrhs])
            assert np.all(err <= tol * scale[:, :nrhs] + 2.0 ** -52), (precision, nrhs)
    a_rp, a_col, a_val = op.assemble()
    assert np.array_equal(a_rp.cpu().numpy(), rp) and np.array_equal(a_col.cpu().numpy(), col)
    dense = torch.zeros(m, dtype=torch.float64, device="cuda")
    dense.index_add_(0, torch.tensor(row, device="cuda"), a_val * xt[0][a_col.long()])
    assert np.all(np.abs(dense.cpu().numpy() - y_o[:, 0]) <= 1e-13 * scale[:, 0])


@pytest.mark.parametrize("kind,n", [("uniform", 3_001), ("blob", 20_003)])
def test_stencil_widened_past_groups(ctx, kind, n):
    """A radius a rounding above two cells: the plan is made for 125 buckets (for
    the eight-lane form alone, or with both lists), and centres just below a
    cell's face have a neighbour three cells on, so it is made again with 343
    and work items only."""
    rng = np.random.default_rng(n)
    pos = cloud(kind, n, 3, rng)
    face = np.arange(3, 13) / 16.0
    pos[:10] = np.stack([face * (1.0 - 1e-13), face + 0.01, face + 0.02], 1)
    pos[10:20] = np.stack([face + 2.0 / 16.0, face + 0.01, face + 0.02], 1)
    low, high, per = [0.0] * 3, [1.0] * 3, [False] * 3
    leaf = 0.999 * n / 4096.0
    cl = ab.CellListOrdered(ctx, low, high, per, leaf)
    cl.update_positions(torch.tensor(pos, device="cuda"))
    oc = oracle.Cells(low, high, per, leaf)
    oc.update(pos.copy(), np.ones(n, np.uint8))
    assert list(oc.grid) == [16] * 3
    r = 2.0 / 16.0 * (1.0 + 5e-10)
    centres = cl.positions()
    q = centres.cpu().numpy()
    rp_o, col_o = oc.search(q, r)
    cell = np.floor(q * 16.0)
    apart = np.abs(np.repeat(cell, np.diff(rp_o), 0) - cell[col_o]).max(1)
    assert apart.max() == 3
    search = ab.Search(cl, centres, r)
    for _ in range(2):  # the handle's plan is made anew
        rp = search.row_ptr().cpu().numpy()
        col = torch.zeros(search.total, dtype=torch.int32, device="cuda")
        search.fill(col)
        assert np.array_equal(rp, rp_o)
        row = np.repeat(np.arange(n), np.diff(rp))
        col = col.cpu().numpy()
        assert np.array_equal(col[np.lexsort((col, row))], col_o[np.lexsort((col_o, row))])
        search.run(cl, centres, r)
    one = torch.zeros(len(col) + 5, dtype=torch.int32, device="cuda")
    assert search.run_fused(cl, centres, r, one) == len(col)
    assert np.array_equal(one.cpu().numpy()[:len(col)], col)
    x = rng.standard_normal((n, 3))
    y_o = oc.sparse_matvec(q, r, (1, 0.5 * r), x)
    scale = oc.sparse_matvec(q, r, (1, 0.5 * r), np.abs(x))
    op = ab.SparseOperator(ctx, cl, centres, r, ab.Kernel.gaussian(0.5 * r))
    y = torch.zeros(3, n, dtype=torch.float64, device="cuda")
    op.apply_colmajor(torch.tensor(x.T.copy(), device="cuda"), y)
    assert np.all(np.abs(y.cpu().numpy().T - y_o) <= 1e-13 * scale)
