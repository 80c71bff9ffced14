"""What a plan reports can be given back: the radices and tiles of every default plan make the
same plan through an explicit split, and so do the tuner's; and the kernels that the
reports name are the ones that run."""
import json

import pytest

import estl_amd

pytestmark = pytest.mark.gpu


def log2s(values):
    return [v.bit_length() - 1 for v in values]


def rebuilt(desc, n, batch, precision, tiles=True):
    return estl_amd.Plan(n, batch, estl_amd.FORWARD, precision, split=log2s([p["radix"] for p in desc["passes"]]),
                         tiles=log2s([p["tile"] for p in desc["passes"]]) if tiles else None)


@pytest.mark.parametrize("precision", [estl_amd.FP32, estl_amd.FP16])
@pytest.mark.parametrize("log2n,batch", [(14, 1), (15, 300), (17, 9), (18, 101), (19, 1), (19, 2), (19, 5), (20, 1),
                                         (20, 2), (20, 3), (21, 1), (23, 1)])
def test_default_plan_round_trip(gpu, precision, log2n, batch):
    n = 1 << log2n
    desc = estl_amd.Plan(n, batch, estl_amd.FORWARD, precision).describe()
    for tiles in (True, False):
        assert rebuilt(desc, n, batch, precision, tiles).describe() == desc


def test_fp16_round_trip_computes_the_same(gpu):
    import torch
    n, batch = 1 << 19, 3
    x = torch.empty(batch, n, dtype=torch.complex64, device=gpu)
    estl_amd.fill_uniform(x, 64)
    x16 = torch.empty(batch, n, 2, dtype=torch.float16, device=gpu)
    sx = torch.empty(batch, dtype=torch.float32, device=gpu)
    estl_amd.pack_fp16(x, x16, sx, n, batch)
    p = estl_amd.Plan(n, batch, estl_amd.FORWARD, estl_amd.FP16)
    got = []
    for q in (p, rebuilt(p.describe(), n, batch, estl_amd.FP16)):
        y16, sy = torch.empty_like(x16), torch.empty_like(sx)
        q.execute_fp16(x16, sx, y16, sy)
        got.append((y16, sy))
    assert torch.equal(got[0][0].view(torch.int16), got[1][0].view(torch.int16)) and torch.equal(got[0][1], got[1][1])


def test_fp16_radix_without_kernel_is_refused_at_creation(gpu):
    """Radix 2^10 in FP16 has tiles of 16 columns and no others, and no caller's split but the
    default plan's."""
    for split, tiles in (([10, 9], None), ([9, 10], [4, 3]), ([9, 10], [4, 5]), ([10, 10], None)):
        with pytest.raises(estl_amd.EstlError):
            estl_amd.Plan(1 << sum(split), 1 if split == [10, 10] else 2, estl_amd.FORWARD, estl_amd.FP16, split=split,
                          tiles=tiles)


@pytest.mark.parametrize("log2n,batch", [(18, 4), (19, 2)])
def test_tuned_fp16_plan_round_trip(gpu, log2n, batch):
    n = 1 << log2n
    report = estl_amd.tune(n, batch, estl_amd.FORWARD, estl_amd.FP16)
    default = estl_amd.Plan(n, batch, estl_amd.FORWARD, estl_amd.FP16).describe()
    assert log2s([p["radix"] for p in default["passes"]]) in [c["plan"] for c in report["candidates"]]
    desc = estl_amd.Plan(n, batch, estl_amd.FORWARD, estl_amd.FP16, flags=estl_amd.FLAG_AUTOTUNE).describe()
    assert rebuilt(desc, n, batch, estl_amd.FP16).describe() == desc
