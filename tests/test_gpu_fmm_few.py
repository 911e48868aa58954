"""FMM products of one to eight right-hand sides (columns packed from several
sibling tiles, offsets split) against the sixteen-column form, for every
order, one level of M2L up to several, tile counts that do not fill a block,
and clustered points (missing children).

Bar: both add the same products of the far field in another order: at most a
few hundred terms of size sum |.| per box, 1e-12 of the largest value.
"""
import pytest
import torch

import aboria_amd as ab

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("n,leaf,clustered", [(150, 20.0, False), (3_001, 16.0, False),
                                              (4_000, 12.0, True)])
def test_few_columns_match_sixteen(ctx, order, n, leaf, clustered):
    print("few", order, n, clustered, flush=True)
    g = torch.Generator(device="cuda").manual_seed(n + order)
    pos = torch.rand(n, 3, generator=g, device="cuda", dtype=torch.float64)
    if clustered:
        pos[: n // 2] = 0.05 + 0.1 * pos[: n // 2] ** 3
    x = 2.0 * torch.rand(16, n, generator=g, device="cuda", dtype=torch.float64) - 1.0
    op = ab.FmmOperator(ctx, pos, [0.0] * 3, [1.0] * 3, leaf, order, ab.Kernel.smooth_inv_r(1e-2))
    ref = op.apply_colmajor(x, torch.zeros_like(x))
    for nrhs in (1, 2, 3, 4, 5, 8, 1):
        y = op.apply_colmajor(x[:nrhs].contiguous(), torch.zeros_like(x[:nrhs]))
        assert (y - ref[:nrhs]).abs().max() <= 1e-12 * ref.abs().max(), nrhs
    y = op.apply_colmajor(x[:3].contiguous(), torch.full_like(x[:3], 0.5))
    assert torch.allclose(y - 0.5, ref[:3], rtol=0, atol=1e-12 * float(ref.abs().max()))
