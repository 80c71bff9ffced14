"""GPU parity of the passes with 32 values per thread (k_pass_wide): each compiled radix and
tile as a first, a middle and a last pass, at the smallest strides its dispatch accepts,
against the FP64 oracle.

Tolerance: relative L2 per row <= 1e-6 * log2(n) for FP32, as for every FP32 transform, and
2^-11 * sqrt(stores) for FP16 storage (one rounding to binary16 for the pack and for each
pass).
"""
import math

import numpy as np
import pytest

import estl_amd
import oracle

pytestmark = pytest.mark.gpu

PLANS = [
    # first passes: S = T, S > T
    ([7, 6], [6, 4]), ([8, 5], [5, 4]), ([8, 6], [6, 4]), ([9, 4], [4, 4]), ([9, 5], [5, 4]), ([10, 4], [4, 4]),
    ([7, 8], [6, 5]), ([9, 9], [5, 4]), ([10, 9], [4, 5]),
    # last passes: A = T columns in all, and more
    ([5, 8], [4, 5]), ([6, 8], [4, 6]), ([4, 9], [4, 4]), ([5, 9], [4, 5]), ([4, 10], [4, 4]), ([9, 10], [4, 4]),
    # middle passes: S = T, S > T
    ([4, 7, 6], [4, 6, 4]), ([4, 8, 5], [4, 5, 4]), ([4, 8, 6], [4, 6, 4]), ([4, 9, 4], [4, 4, 4]),
    ([4, 9, 5], [4, 5, 4]), ([4, 10, 4], [4, 4, 4]), ([4, 9, 7], [4, 5, 5]),
    # the default plans that use them
    (None, None),
]


def sizes(split):
    return [1 << sum(split)] if split else [1 << 15, 1 << 18, 1 << 19, 1 << 20]


@pytest.mark.parametrize("split,tiles", PLANS)
@pytest.mark.parametrize("direction", [estl_amd.FORWARD, estl_amd.BACKWARD])
def test_fp32(gpu, split, tiles, direction):
    import torch
    for n in sizes(split):
        for batch, in_place in ((1, False), (3, True), (4, False)):
            x = torch.empty(batch, n, dtype=torch.complex64, device=gpu)
            estl_amd.fill_uniform(x, 95)
            want = oracle.fft64(x.cpu().numpy(), direction)
            p = estl_amd.Plan(n, batch, direction, split=split, tiles=tiles)
            y = x if in_place else torch.empty_like(x)
            p.execute(x, y)
            torch.cuda.synchronize()
            got = y.cpu().numpy()
            for r in range(batch):
                assert oracle.rel_l2(got[r], want[r]) <= 1e-6 * math.log2(n), (n, batch, r)


@pytest.mark.parametrize("split,tiles", [p for p in PLANS if not p[0] or max(p[0]) <= 9])
def test_fp16_storage(gpu, split, tiles):
    import torch
    for n in sizes(split):
        batch = 3
        x = torch.empty(batch, n, dtype=torch.complex64, device=gpu)
        estl_amd.fill_uniform(x, 96)
        want = oracle.fft64(x.cpu().numpy(), estl_amd.FORWARD)
        x16 = torch.empty(batch * n * 2, dtype=torch.float16, device=gpu)
        y16 = torch.empty_like(x16)
        sx = torch.empty(batch, dtype=torch.float32, device=gpu)
        sy = torch.empty_like(sx)
        estl_amd.pack_fp16(x, x16, sx, n, batch)
        p = estl_amd.Plan(n, batch, estl_amd.FORWARD, estl_amd.FP16, split=split, tiles=tiles)
        p.execute_fp16(x16, sx, y16, sy)
        torch.cuda.synchronize()
        got = y16.cpu().numpy().astype(np.float64).reshape(batch, n, 2)
        got = (got[..., 0] + 1j * got[..., 1]) * sy.cpu().numpy().astype(np.float64)[:, None]
        for r in range(batch):
            assert oracle.rel_l2(got[r], want[r]) <= 2.0 ** -11 * math.sqrt(1 + p.launches()), (n, r)


def test_fp16_split_radix_stays_bounded(gpu):
    """An FP16 split of a caller's keeps to radices of at most 2^9."""
    with pytest.raises(estl_amd.EstlError):
        estl_amd.Plan(1 << 20, 1, estl_amd.FORWARD, estl_amd.FP16, split=[10, 10])
