"""Every size class of the uneven batch (rows up to 2^13, two passes of 16 values per thread up
to 2^16, of 32 above), against the FP64 oracle: relative L2 <= 1e-6 * log2(n)."""
import math

import pytest

import estl_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log2n", list(range(12, 21)))
@pytest.mark.parametrize("direction", [estl_amd.FORWARD, estl_amd.BACKWARD])
def test_size_class(gpu, log2n, direction):
    import torch
    sizes = [1 << log2n, 256, 1 << log2n, 1 << log2n]
    x = torch.empty(sum(sizes), dtype=torch.complex64, device=gpu)
    estl_amd.fill_uniform(x, 98)
    y = torch.empty_like(x)
    estl_amd.UnevenBatch(sizes, direction=direction).execute(x, y)
    torch.cuda.synchronize()
    xh, yh, off = x.cpu().numpy(), y.cpu().numpy(), 0
    for n in sizes:
        want = oracle.fft64(xh[off:off + n], direction)
        assert oracle.rel_l2(yh[off:off + n], want) <= 1e-6 * math.log2(n), n
        off += n
