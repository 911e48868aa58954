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
    other_bits = False
    for nrhs in (1, 2, 3, 4, 5, 8, 1):
        y = op.apply_colmajor(x[:nrhs].contiguous(), torch.zeros_like(x[:nrhs]))
        assert (y - ref[:nrhs]).abs().max() <= 1e-12 * ref.abs().max(), nrhs
        other_bits = other_bits or not torch.equal(y, ref[:nrhs])
    # the other kernel did run: thousands of sums in another order
    assert other_bits or n == 150
    y = op.apply_colmajor(x[:3].contiguous(), torch.full_like(x[:3], 0.5))
    assert torch.allclose(y - 0.5, ref[:3], rtol=0, atol=1e-12 * float(ref.abs().max()))


def test_few_columns_limit(ctx):
    """Where the packed form's buffers (2 GB at most) hold one column only, one
    column takes it and two and more take the sixteen-column form."""
    n = 50_000
    g = torch.Generator(device="cuda").manual_seed(1)
    pos = torch.rand(n, 3, generator=g, device="cuda", dtype=torch.float64)
    x = 2.0 * torch.rand(16, n, generator=g, device="cuda", dtype=torch.float64) - 1.0
    op = ab.FmmOperator(ctx, pos, [0.0] * 3, [1.0] * 3, 2.0, 8, ab.Kernel.smooth_inv_r(1e-2))
    # 8 splits of 8 children per parent of the widest level, all nodes, 512 rows
    nodes = op.info["n_nodes"]
    assert op.info["levels"] >= 5 and 2 * 8 * 512 * 8 * (nodes // 2) > 2 << 30
    ref = op.apply_colmajor(x, torch.zeros_like(x))
    for nrhs in (1, 2, 8):
        y = op.apply_colmajor(x[:nrhs].contiguous(), torch.zeros_like(x[:nrhs]))
        assert (y - ref[:nrhs]).abs().max() <= 1e-12 * ref.abs().max(), nrhs
        assert torch.equal(y, ref[:nrhs]) == (nrhs > 1)


def test_few_columns_captured():
    """A captured apply repeats the eager one's bits; one captured before any
    apply of few columns takes the sixteen-column form, which needs no new
    buffers."""
    n = 3_001
    g = torch.Generator(device="cuda").manual_seed(2)
    pos = torch.rand(n, 3, generator=g, device="cuda", dtype=torch.float64)
    x = 2.0 * torch.rand(16, n, generator=g, device="cuda", dtype=torch.float64) - 1.0
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        c = ab.Context(0, stream)
        for first in (2, 16):
            op = ab.FmmOperator(c, pos, [0.0] * 3, [1.0] * 3, 16.0, 4, ab.Kernel.smooth_inv_r(1e-2))
            ref = op.apply_colmajor(x[:first].contiguous(), torch.zeros_like(x[:first]))[:2]
            y = torch.zeros_like(x[:2])
            x2 = x[:2].contiguous()
            stream.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                op.apply_colmajor(x2, y)
            for _ in range(3):
                y.zero_()
                graph.replay()
                stream.synchronize()
                assert torch.equal(y, ref)
                op.apply_colmajor(x[:1].contiguous(), torch.zeros_like(x[:1]))
            del graph, op
        c.close()
