"""GPU parity of the plans that a caller gets without asking for a split, at the loads where
the planner's rules change (the last radix, two passes or three, tiles of 32 values per
thread or 16), on a few rows of each batch; and of 2-D plans whose columns take one wide
pass, in place or not.

Tolerances as everywhere: relative L2 <= 1e-6 * log2(values) for FP32, 2^-11 * sqrt(stores)
for FP16 storage (one rounding to binary16 for the pack and for each pass).
"""
import math

import numpy as np
import pytest

import estl_amd
import oracle

pytestmark = pytest.mark.gpu


def rows_of(batch):
    return sorted({0, 1 % batch, batch // 2, batch - 1})


@pytest.mark.parametrize("log2n,batch", [(14, 512), (15, 255), (15, 256), (16, 64), (16, 128), (17, 64), (18, 32),
                                         (19, 3), (19, 4), (20, 1), (20, 2), (21, 2), (22, 2)])
@pytest.mark.parametrize("direction", [estl_amd.FORWARD, estl_amd.BACKWARD])
def test_fp32(gpu, log2n, batch, direction):
    import torch
    n = 1 << log2n
    x = torch.empty(batch, n, dtype=torch.complex64, device=gpu)
    estl_amd.fill_uniform(x, 61)
    y = torch.empty_like(x)
    estl_amd.Plan(n, batch, direction).execute(x, y)
    torch.cuda.synchronize()
    for r in rows_of(batch):
        want = oracle.fft64(x[r].cpu().numpy(), direction)
        assert oracle.rel_l2(y[r].cpu().numpy(), want) <= 1e-6 * log2n, r


@pytest.mark.parametrize("log2n,batch", [(14, 64), (15, 32), (15, 33), (16, 15), (16, 16), (17, 8), (18, 4), (19, 1),
                                         (19, 2), (20, 1), (20, 2), (21, 1), (21, 2), (22, 1), (24, 1)])
def test_fp16_storage(gpu, log2n, batch):
    import torch
    n = 1 << log2n
    x = torch.empty(batch, n, dtype=torch.complex64, device=gpu)
    estl_amd.fill_uniform(x, 62)
    x16 = torch.empty(batch, n, 2, dtype=torch.float16, device=gpu)
    y16 = torch.empty_like(x16)
    sx = torch.empty(batch, dtype=torch.float32, device=gpu)
    sy = torch.empty_like(sx)
    estl_amd.pack_fp16(x, x16, sx, n, batch)
    p = estl_amd.Plan(n, batch, estl_amd.FORWARD, estl_amd.FP16)
    p.execute_fp16(x16, sx, y16, sy)
    torch.cuda.synchronize()
    for r in rows_of(batch):
        want = oracle.fft64(x[r].cpu().numpy(), estl_amd.FORWARD)
        got = torch.view_as_complex(y16[r].double() * sy[r].double()).cpu().numpy()
        assert oracle.rel_l2(got, want) <= 2.0 ** -11 * math.sqrt(1 + p.launches()), r


@pytest.mark.parametrize("nx,ny,batch", [(8192, 128, 2), (16384, 256, 1), (8192, 512, 2), (64, 128, 129),
                                         (1024, 512, 4), (128, 8192, 2)])
@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("direction", [estl_amd.FORWARD, estl_amd.BACKWARD])
def test_plan2d(gpu, nx, ny, batch, in_place, direction):
    import torch
    x = torch.empty(batch, ny, nx, dtype=torch.complex64, device=gpu)
    estl_amd.fill_uniform(x, 63)
    xh = x[[0, batch - 1]].cpu().numpy().astype(np.complex128)
    y = x if in_place else torch.empty_like(x)
    estl_amd.Plan2D(nx, ny, batch, direction).execute(x, y)
    torch.cuda.synchronize()
    for b, at in enumerate((0, batch - 1)):
        rows = oracle.fft64(xh[b], direction)
        want = oracle.fft64(np.ascontiguousarray(rows.T), direction).T
        assert oracle.rel_l2(y[at].cpu().numpy(), want) <= 1e-6 * math.log2(nx * ny), at
