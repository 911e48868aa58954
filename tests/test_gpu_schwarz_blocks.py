"""Schwarz factorisation at the edges of its 64-wide blocks, against a dense
solve, and preconditioners that take over memory of earlier ones."""
import numpy as np
import pytest
import torch

import aboria_amd as ab

pytestmark = pytest.mark.gpu


def cells(ctx, pos, n_leaf):
    d = pos.shape[1]
    cl = ab.CellListOrdered(ctx, [0.0] * d, [1.0] * d, [False] * d, n_leaf)
    cl.update_positions(torch.tensor(pos, device="cuda"))
    return cl


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 200, 320])
def test_single_domain_sizes(ctx, n):
    """One bucket: the preconditioner is the inverse.  Bound: backward error of
    a Cholesky solve, (8 n eps) cond(A) of the solution."""
    print("domain", n, flush=True)
    rng = np.random.default_rng(n)
    cl = cells(ctx, rng.random((n, 2)), 4.0 * n)
    p = cl.positions().cpu().numpy()
    a = np.exp(-((p[:, None] - p[None]) ** 2).sum(-1) / 0.05 ** 2) + 0.1 * np.eye(n)
    sw = ab.SchwartzPreconditioner(ctx, cl, ab.Kernel.gaussian(0.05), 0.0, 0.1)
    b = rng.standard_normal(n)
    x = sw.solve(torch.tensor(b, device="cuda")).cpu().numpy()
    ref = np.linalg.solve(a, b)
    assert np.linalg.norm(x - ref) <= 8 * n * 2.0 ** -52 * np.linalg.cond(a) * np.linalg.norm(ref)


@pytest.mark.parametrize("dim,n,leaf", [(1, 700, 23.0), (2, 3_000, 9.0), (2, 3_000, 40.0),
                                        (3, 2_000, 20.0)])
def test_domains_against_dense_solves(ctx, dim, n, leaf):
    """Interior rows of every domain's inverse (interior counts below and above
    64, domains of several blocks) against numpy on the same lists; the
    second preconditioner is built from what the first gave back and the
    third differs from both in size."""
    rng = np.random.default_rng(dim * n)
    for size in (n, n, n // 3):
        print("domains", dim, size, leaf, flush=True)
        cl = cells(ctx, rng.random((size, dim)), leaf)
        p = cl.positions().cpu().numpy()
        sw = ab.SchwartzPreconditioner(ctx, cl, ab.Kernel.gaussian(0.05), 0.3, 0.1)
        b = rng.standard_normal(size)
        x = sw.solve(torch.tensor(b, device="cuda")).cpu().numpy()
        off, idx, nint = sw.domains()
        for d in range(0, len(nint), max(1, len(nint) // 20)):
            i = idx[off[d]:off[d + 1]]
            r2 = ((p[i][:, None] - p[i][None]) ** 2).sum(-1)
            a = np.exp(-r2 / 0.05 ** 2) * (r2 <= 0.3 ** 2) + 0.1 * np.eye(len(i))
            ref = np.linalg.solve(a, b[i])
            err = np.abs(x[i[:nint[d]]] - ref[:nint[d]]).max()
            assert err <= 8 * len(i) * 2.0 ** -52 * np.linalg.cond(a) * np.linalg.norm(ref)
        del sw


@pytest.mark.parametrize("n", [511, 577, 1_024, 1_536, 1_537, 2_048, 2_049, 2_111])
def test_panel_sizes(ctx, n):
    """One domain of one 512-column panel of the factorisation and of several, in
    the Cholesky form and in the signed form of a batch.  Bound as above."""
    print("panel", n, flush=True)
    rng = np.random.default_rng(n)
    pos, b = rng.random((n, 2)), rng.standard_normal(n)
    cl = cells(ctx, pos, 4.0 * n)
    batch = ab.DenseBatchOperator(ctx, [0, n], torch.tensor(pos, device="cuda"),
                                  ab.Kernel.gaussian(0.05))
    for p, sw in ((cl.positions().cpu().numpy(),
                   ab.SchwartzPreconditioner(ctx, cl, ab.Kernel.gaussian(0.05), 0.0, 0.1)),
                  (pos, ab.SchwartzPreconditioner.for_dense_batch(
                      batch, [0.0] * 2, [1.0] * 2, 4.0 * n, 0.1))):
        assert sw.info["n_domains"] == 1 and sw.info["failed_domains"] == 0
        a = np.exp(-((p[:, None] - p[None]) ** 2).sum(-1) / 0.05 ** 2) + 0.1 * np.eye(n)
        x = sw.solve(torch.tensor(b, device="cuda")).cpu().numpy()
        ref = np.linalg.solve(a, b)
        bound = 8 * n * 2.0 ** -52 * np.linalg.cond(a) * np.linalg.norm(ref)
        assert np.linalg.norm(x - ref) <= bound
