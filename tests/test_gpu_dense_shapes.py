"""Rectangular dense apply at the edges of its column ranges (32), staged
chunks (128), row blocks (256) and right-hand-side groups (1, 4, 8, 16), for
every profile, against a plain FP64 sum.

Bar: |y - ref| <= (ncols + 64) eps sum_j |K_ij x_j| in FP64 (each term rounded
to within a few ulp, the sum of ncols terms in any order), 2e-6 of the same
scale in FP32-compensated.
"""
import numpy as np
import pytest
import torch

import aboria_amd as ab

pytestmark = pytest.mark.gpu

KERNELS = {
    "constant": (ab.Kernel.constant(w0=1.0), lambda r2: torch.ones_like(r2)),
    "gaussian": (ab.Kernel.gaussian(0.2), lambda r2: torch.exp(-r2 / 0.04)),
    "wendland": (ab.Kernel.wendland_c2(0.7),
                 lambda r2: (1 - r2.sqrt() / 0.7).clamp(min=0) ** 4 * (4 * r2.sqrt() / 0.7 + 1)),
    "multiquadric": (ab.Kernel.multiquadric(0.1), lambda r2: (r2 + 0.01).sqrt()),
    "inverse": (ab.Kernel.smooth_inv_r(0.05), lambda r2: 1 / (r2.sqrt() + 0.05)),
}


@pytest.mark.parametrize("precision", [ab.FP64, ab.FP32_COMPENSATED])
@pytest.mark.parametrize("nrows,ncols,nrhs,dim,name", [
    (1, 1, 1, 3, "gaussian"), (255, 31, 2, 2, "inverse"), (257, 33, 4, 1, "multiquadric"),
    (256, 129, 5, 3, "wendland"), (1000, 128, 8, 2, "constant"), (77, 4097, 9, 3, "gaussian"),
    (300, 255, 16, 2, "multiquadric"), (513, 1000, 17, 3, "inverse"), (9, 0, 1, 2, "gaussian"),
    (60_000, 65, 1, 2, "wendland"),
])
def test_dense_apply_shapes(ctx, nrows, ncols, nrhs, dim, name, precision):
    g = torch.Generator(device="cuda").manual_seed(nrows * 7 + ncols)
    rand = lambda *s: torch.rand(*s, generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
    rows, cols, x = rand(nrows, dim), rand(ncols, dim), rand(nrhs, ncols) - 0.5
    kernel, phi = KERNELS[name]
    y = torch.full((nrhs, nrows), 0.25, dtype=torch.float64, device="cuda")
    ab.dense_apply(ctx, rows, cols, kernel, x, y, precision)
    f = phi((rows[:, None] - cols[None]).square().sum(-1))
    ref, scale = x @ f.t(), x.abs() @ f.t()
    tol = (ncols + 64) * 2.0 ** -52 if precision == ab.FP64 else 2e-6
    assert torch.all((y - 0.25 - ref).abs() <= tol * scale + 2.0 ** -52)


def test_dense_apply_captured(ctx):
    """A captured apply of a shape that splits only when it is not captured:
    every replay adds K x, whatever the context does in between."""
    g = torch.Generator(device="cuda").manual_seed(3)
    rand = lambda *s: torch.rand(*s, generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
    rows, cols, x = rand(500, 3), rand(700, 3), rand(2, 700) - 0.5
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        c = ab.Context(0, stream)
        kernel = ab.Kernel.gaussian(0.2)
        y = torch.zeros(2, 500, dtype=torch.float64, device="cuda")
        ref = ab.dense_apply(c, rows, cols, kernel, x)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            ab.dense_apply(c, rows, cols, kernel, x, y)
        for k in range(1, 4):
            graph.replay()
            big = ab.dense_apply(c, rand(4000 * k, 3), rand(5000, 3), kernel, rand(3, 5000))
            stream.synchronize()
            assert torch.allclose(y, k * ref, rtol=1e-12, atol=1e-12)
            assert torch.isfinite(big).all()
        c.close()


@pytest.mark.parametrize("nrows,ncols,nrhs", [(300, 50_000, 2), (40, 9_000, 16)])
def test_captured_split_keeps_its_buffer(ctx, nrows, ncols, nrhs):
    """A captured apply that splits its columns (ranges of 2,048 and more) while
    later calls need larger buffers of the context: no buffer that the graph
    knows is freed, and every replay adds K x.  Bar: each replay's sum and ref
    are within ncols roundings of the exact one."""
    g = torch.Generator(device="cuda").manual_seed(nrows)
    rand = lambda *s: torch.rand(*s, generator=g, device="cuda", dtype=torch.float64)  # noqa: E731
    rows, cols, x = rand(nrows, 3), rand(ncols, 3), rand(nrhs, ncols) - 0.5
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        c = ab.Context(0, stream)
        kernel = ab.Kernel.gaussian(0.2)
        y = torch.zeros(nrhs, nrows, dtype=torch.float64, device="cuda")
        ref = ab.dense_apply(c, rows, cols, kernel, x)
        scale = ab.dense_apply(c, rows, cols, kernel, x.abs())
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            ab.dense_apply(c, rows, cols, kernel, x, y)
        # fine splits of up to 32 MiB, then a coarse one of 82 MiB
        shapes = [(5_000, 4_001, 1), (4_000, 5_000, 3), (20_000, 65_536, 16), (300, 60_000, 4)]
        for k, (m, n, r) in enumerate(shapes, 1):
            print("replay", k, flush=True)
            big = ab.dense_apply(c, rand(m, 3), rand(n, 3), kernel, rand(r, n))
            stream.synchronize()
            graph.replay()
            stream.synchronize()
            assert torch.all((y - k * ref).abs() <= (k + 1) * (ncols + 64) * 2.0 ** -52 * scale)
            assert torch.isfinite(big).all()
        del graph
        c.close()
