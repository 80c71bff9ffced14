"""The FP16 pack on both sides of the line where it takes eight values per thread (2^22 values
in all), with a ragged last workgroup.  Exact: the scale is the largest |re| or |im| (1 for
zeros) and the stored values are x / scale rounded to binary16."""
import pytest

import estl_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log2n,batch", [(7, 32767), (7, 32768), (7, 32769), (3, 2 ** 19 + 5), (15, 127), (15, 129),
                                         (18, 15), (18, 16), (22, 1), (1, 2 ** 21 - 1), (1, 2 ** 21 + 1)])
def test_pack_is_exact(gpu, log2n, batch):
    import torch
    n = 1 << log2n
    x = torch.empty(batch, n, 2, dtype=torch.float32, device=gpu)
    estl_amd.fill_uniform(x, 97)
    x *= torch.tensor([1.0, 1e-5, 3e4], device=gpu)[torch.arange(batch, device=gpu) % 3][:, None, None]
    x[batch // 2] = 0.0
    x[0, n - 1, 1] = -70000.0
    scale = x.abs().amax(dim=(1, 2))
    scale[scale == 0] = 1.0
    want = (x / scale[:, None, None]).to(torch.float16)
    x16 = torch.full((batch * n * 2 + 8,), 5.0, dtype=torch.float16, device=gpu)
    s = torch.full((batch + 1,), -1.0, device=gpu)
    estl_amd.pack_fp16(torch.view_as_complex(x), x16, s, n, batch)
    torch.cuda.synchronize()
    assert torch.equal(s[:batch], scale) and s[batch].item() == -1.0
    assert torch.equal(x16[:batch * n * 2].view(batch, n, 2), want)
    assert bool((x16[batch * n * 2:] == 5.0).all())
