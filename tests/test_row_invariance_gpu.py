"""Which results do not depend on what else a call computes, bit for bit: rows of up to 2^13
values in batches of any size, rows of any length through one split and its tiles, the row
convolutions and overlap-save windows of one length, and the transforms of an uneven batch, which are
those of the rows plans up to 2^13 and of the even split above.  (A default plan above 2^13
is chosen by n and batch, and promises its error bound only.)"""
import pytest

import estl_amd

pytestmark = pytest.mark.gpu


def run(plan, x):
    import torch
    y = torch.empty_like(x)
    plan.execute(x, y)
    return torch.view_as_real(y)


def rows(gpu, batch, n, seed=71):
    import torch
    x = torch.empty(batch, n, dtype=torch.complex64, device=gpu)
    estl_amd.fill_uniform(x, seed)
    return x


@pytest.mark.parametrize("log2n", [1, 4, 5, 8, 9, 11, 12, 13])
def test_rows(gpu, log2n):
    import torch
    n = 1 << log2n
    x = rows(gpu, 301, n)
    whole = run(estl_amd.Plan(n, 301), x)
    for at, count in ((0, 1), (7, 3), (300, 1)):
        part = run(estl_amd.Plan(n, count), x[at:at + count].clone())
        assert torch.equal(part, whole[at:at + count]), (n, at)


@pytest.mark.parametrize("split,tiles", [([7, 7], [6, 5]), ([7, 8], [6, 5]), ([9, 9], [5, 5]), ([9, 10], [5, 4]),
                                         ([6, 7, 7], [6, 6, 4])])
def test_explicit_splits(gpu, split, tiles):
    import torch
    n, batch = 1 << sum(split), 9
    x = rows(gpu, batch, n)
    whole = run(estl_amd.Plan(n, batch, split=split, tiles=tiles), x)
    for at in (0, 4, 8):
        part = run(estl_amd.Plan(n, 1, split=split, tiles=tiles), x[at:at + 1].clone())
        assert torch.equal(part, whole[at:at + 1]), at


@pytest.mark.parametrize("n,k", [(2 ** 9, 33), (2 ** 10, 33), (2 ** 11, 300), (2 ** 12, 300), (2 ** 13, 33),
                                 (2 ** 15, 8000), (2 ** 14, 100)])
def test_convolution_rows(gpu, n, k):
    """Pairs of rows share a transform: the pairs of a longer batch come out as alone."""
    import torch
    x = torch.empty(40, n, device=gpu)
    h = torch.empty(k, device=gpu)
    estl_amd.fill_uniform(x, 72)
    estl_amd.fill_uniform(h, 73)

    def conv(part):
        c = estl_amd.Convolution(n, part.shape[0])
        c.set_filter(h)
        y = torch.empty_like(part)
        c.execute(part, y)
        return y

    whole = conv(x)
    for at, count in ((0, 2), (6, 4), (38, 2)):
        assert torch.equal(conv(x[at:at + count].clone()), whole[at:at + count]), (n, at)


@pytest.mark.parametrize("log2n", [4, 8, 11, 12, 13, 14, 15, 16, 17, 18, 19, 20])
def test_uneven_batch(gpu, log2n):
    import torch
    n = 1 << log2n
    x = rows(gpu, 3, n)
    flat = torch.cat([x[0], rows(gpu, 1, 256)[0], x[1], x[2]])
    y = torch.empty_like(flat)
    estl_amd.UnevenBatch([n, 256, n, n]).execute(flat, y)
    if log2n <= 13:
        plan = estl_amd.Plan(n, 3)
    elif log2n <= 16:  # 16 values per thread, whatever the tiles of a plan
        plan = estl_amd.Plan(n, 3, split=[log2n // 2, log2n - log2n // 2], tiles=[3, 3])
    else:              # 32 values per thread
        b = log2n // 2
        plan = estl_amd.Plan(n, 3, split=[b, log2n - b], tiles=[14 - b, 14 - (log2n - b)])
        assert plan.describe()["kernel"] == "k_pass_wide"
    want = run(plan, x)
    got = torch.view_as_real(y)
    for r, at in enumerate((0, n + 256, 2 * n + 256)):
        assert torch.equal(got[at:at + n], want[r]), r
