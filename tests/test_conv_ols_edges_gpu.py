"""GPU parity of k_conv_ols where its stores begin and end: windows whose outputs the
rotation carries past the row's end (one store piece or two), a short last window, a lone
last window, the longest filters, in both storage types.

Tolerance: FP32 relative L2 per row <= 2e-6 * log2(n), as for every FP32 convolution; FP16
storage 2^-11 * 4, one binary16 store of outputs relative to their L1 bound (the inputs are
compared as stored).
"""
import math

import numpy as np
import pytest

import estl_amd
import oracle

pytestmark = pytest.mark.gpu

CORR, CENTER = estl_amd.CONV_CORRELATE, estl_amd.CONV_CENTER


def reference(x, h, flags):
    n, k = x.shape[1], len(h)
    hp = np.zeros(n)
    np.add.at(hp, np.arange(k) % n, h.astype(np.float64))
    if flags & CENTER:
        hp = np.roll(hp, -((k + 1) // 2))
    spec = np.fft.fft(hp)
    return np.real(np.fft.ifft(np.fft.fft(x.astype(np.float64), axis=1) * (np.conj(spec) if flags & CORR else spec),
                               axis=1))


@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("n,rows,k,flags", [
    (2 ** 14, 1, 2, CENTER),           # rotation by one
    (2 ** 14, 2, 33, CENTER | CORR),   # rotated forward
    (2 ** 14, 3, 4097, CENTER),        # a lone last window, rotated
    (2 ** 14, 5, 129, 0),
    (2 ** 15, 1, 8193, CENTER | CORR),  # 2^14 windows, the longest filter
    (2 ** 15, 3, 8192, CENTER),
    (2 ** 17, 3, 4095, CENTER),
    (2 ** 18, 2, 6001, CORR),
])
def test_window_edges(gpu, fp16, n, rows, k, flags):
    import torch
    x = oracle.fill_uniform(rows * n, 92).astype(np.float32).reshape(rows, n)
    h = oracle.fill_uniform(k, 93).astype(np.float32)
    dx, dh = torch.from_numpy(x).to(gpu).reshape(-1), torch.from_numpy(h).to(gpu)
    # values before and after the rows: nothing outside them is written
    buf = torch.full((rows * n + 2,), 7.0, device=gpu, dtype=torch.float16 if fp16 else torch.float32)
    out = buf[1:1 + rows * n]
    c = estl_amd.Convolution(n, rows, flags, precision=estl_amd.FP16 if fp16 else estl_amd.FP32)
    c.set_filter(dh)
    if fp16:
        x16 = torch.empty(rows * n, dtype=torch.float16, device=gpu)
        sx = torch.empty(rows, device=gpu)
        sy = torch.empty_like(sx)
        estl_amd.pack_fp16(dx, x16, sx, n // 2, rows)
        c.execute_fp16(x16, sx, out, sy)
        x = (x16.float().view(rows, n) * sx[:, None]).cpu().numpy()
        y = (out.float().view(rows, n) * sy[:, None]).cpu().numpy()
    else:
        c.execute(dx, out)
        y = out.cpu().numpy().reshape(rows, n)
    assert buf[0].item() == 7.0 and buf[-1].item() == 7.0
    ref = reference(x, h, flags)
    for r in range(rows):
        e = oracle.rel_l2(y[r].astype(np.float64), ref[r])
        assert e <= (2.0 ** -11 * 4 if fp16 else 2e-6 * math.log2(n)), (r, e)


@pytest.mark.parametrize("log2n", [10, 11, 12, 13])
@pytest.mark.parametrize("rows", [1, 3, 15, 17])   # a lone row, ragged workgroups
def test_fp16_rows(gpu, log2n, rows):
    """The row convolutions on binary16 rows, ragged workgroups included."""
    import torch
    n, k = 1 << log2n, 33
    x = oracle.fill_uniform(rows * n, 94).astype(np.float32).reshape(rows, n)
    h = oracle.fill_uniform(k, 95).astype(np.float32)
    c = estl_amd.Convolution(n, rows, CORR, precision=estl_amd.FP16)
    c.set_filter(torch.from_numpy(h).to(gpu))
    x16 = torch.empty(rows * n, dtype=torch.float16, device=gpu)
    sx = torch.empty(rows, device=gpu)
    estl_amd.pack_fp16(torch.from_numpy(x).to(gpu).reshape(-1), x16, sx, n // 2, rows)
    buf = torch.full((rows * n + 2,), 7.0, device=gpu, dtype=torch.float16)
    sy = torch.full((rows + 1,), -1.0, device=gpu)
    c.execute_fp16(x16, sx, buf[1:1 + rows * n], sy)
    assert buf[0].item() == 7.0 and buf[-1].item() == 7.0 and sy[rows].item() == -1.0
    y = (buf[1:-1].float().view(rows, n) * sy[:rows, None]).cpu().numpy()
    ref = reference((x16.float().view(rows, n) * sx[:, None]).cpu().numpy(), h, CORR)
    for r in range(rows):
        assert oracle.rel_l2(y[r].astype(np.float64), ref[r]) <= 2.0 ** -11 * 4, r
