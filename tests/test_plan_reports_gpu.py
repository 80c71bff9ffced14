"""What a plan reports can be given back: the radices and tiles of every default plan make the
same plan through an explicit split, and so do the tuner's; and the kernels that the
reports name are the ones that run."""
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


@pytest.mark.parametrize("precision,plain", [(estl_amd.FP32, "k_fft_pass"), (estl_amd.FP16, "k_fft_pass_h")])
def test_reports_name_the_kernels_that_run(gpu, precision, plain):
    """The wide kernel has radices 2^7 .. 2^10 in its own tiles; every other pass is the plain
    one's.  describe() and the profile's lines say which runs each pass."""
    for split, tiles, want in [([9, 9], [5, 5], ["k_pass_wide"] * 2), ([9, 9], [3, 3], [plain] * 2),
                               ([6, 8], [6, 5], [plain, "k_pass_wide"])]:
        p = estl_amd.Plan(1 << sum(split), 4, estl_amd.FORWARD, precision, split=split, tiles=tiles)
        desc = p.describe()
        assert [q["kernel"] for q in desc["passes"]] == want
        assert desc["kernel"] == ", ".join(dict.fromkeys(want))
        info = [k["info"] for k in p.profile(1)["kernels"]]
        assert [i.split(",")[0] for i in info] == want
    names = [q["kernel"] for q in estl_amd.Plan(1 << 20, 33, estl_amd.FORWARD, precision).describe()["passes"]]
    assert names == ["k_pass_wide"] * 2


def test_reports_name_the_rows_kernels(gpu):
    for precision, flags, want in [(estl_amd.FP32, 0, "k_fft_rows"), (estl_amd.FP16, 0, "k_fft_rows_h"),
                                   (estl_amd.FP32, estl_amd.FLAG_PLANAR, "k_fft_rows_planar")]:
        p = estl_amd.Plan(1 << 10, 64, estl_amd.FORWARD, precision, flags=flags)
        assert p.describe()["kernel"] == want
        assert p.profile(1)["kernels"][0]["info"].split(",")[0] == want
