"""The FP16 pack at the edges of its kernels: one launch for transforms of 2^8 .. 2^14
values (k_pack_rows, whose workgroups take several short transforms), separate maximum and
conversion below and above.  Exact: the scale is the largest |re| or |im| (1 for zeros) and
the stored values are x / scale rounded to binary16.
"""
import numpy as np
import pytest

import estl_amd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log2n", [1, 7, 8, 9, 11, 12, 13, 14, 15, 17])
@pytest.mark.parametrize("batch", [1, 3, 17])
def test_pack_is_exact(gpu, log2n, batch):
    import torch
    n = 1 << log2n
    x = oracle.fill_uniform(batch * n * 2, 97).astype(np.float32).reshape(batch, n, 2)
    x *= np.array([1.0, 1e-5, 3e4], np.float32)[np.arange(batch) % 3][:, None, None]
    x[batch // 2] = 0.0                       # a transform of zeros: scale 1
    x[0, n - 1, 1] = -np.float32(70000.0)     # the peak in the last value
    scale = np.abs(x).max(axis=(1, 2))
    scale[scale == 0] = 1.0
    want = (x / scale[:, None, None]).astype(np.float16)
    dx = torch.view_as_complex(torch.from_numpy(x).to(gpu))
    x16 = torch.full((batch * n * 2 + 8,), 5.0, dtype=torch.float16, device=gpu)
    s = torch.full((batch + 1,), -1.0, device=gpu)
    estl_amd.pack_fp16(dx, x16, s, n, batch)
    torch.cuda.synchronize()
    assert np.array_equal(s.cpu().numpy()[:batch], scale) and s[batch].item() == -1.0
    assert np.array_equal(x16.cpu().numpy()[:batch * n * 2].reshape(batch, n, 2), want)
    assert bool((x16[batch * n * 2:] == 5.0).all())
