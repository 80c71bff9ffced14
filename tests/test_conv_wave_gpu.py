"""GPU parity of the convolutions that keep 32 values per thread (k_conv_wave for rows of
2^10 .. 2^13 values, k_conv_ols for longer ones) at the sizes where their indexing can go
wrong, against the convolution theorem in FP64.

Tolerance: relative L2 per row <= 2e-6 * log2(n), as for every FP32 convolution (a forward
and an inverse FP32 transform plus a complex multiply between them).
"""
import math

import numpy as np
import pytest

import estl_amd
import oracle

pytestmark = pytest.mark.gpu

CORR, CENTER = estl_amd.CONV_CORRELATE, estl_amd.CONV_CENTER


def check(gpu, n, rows, k, flags):
    import torch
    x = oracle.fill_uniform(rows * n, 90).astype(np.float32).reshape(rows, n)
    h = oracle.fill_uniform(k, 91).astype(np.float32)
    hp = np.zeros(n)
    np.add.at(hp, np.arange(k) % n, h.astype(np.float64))
    if flags & CENTER:
        hp = np.roll(hp, -((k + 1) // 2))
    spec = np.fft.fft(hp)
    if flags & CORR:
        spec = np.conj(spec)
    ref = np.real(np.fft.ifft(np.fft.fft(x.astype(np.float64), axis=1) * spec, axis=1))
    c = estl_amd.Convolution(n, rows, flags)
    # one float before and after the rows: nothing outside them is written
    buf = torch.full((rows * n + 2,), 7.0, device=gpu)
    c.set_filter(torch.from_numpy(h).to(gpu))
    dx = torch.from_numpy(x).to(gpu).reshape(-1)
    c.execute(dx, buf[1:1 + rows * n])
    torch.cuda.synchronize()
    assert buf[0].item() == 7.0 and buf[-1].item() == 7.0
    y = buf[1:-1].cpu().numpy().reshape(rows, n).astype(np.float64)
    for r in range(rows):
        e = oracle.rel_l2(y[r], ref[r])
        assert e <= 2e-6 * math.log2(n), (r, e)


@pytest.mark.parametrize("log2n", [10, 11, 12, 13])
@pytest.mark.parametrize("rows", [1, 2, 15, 17])   # a lone row, one pair, ragged workgroups
@pytest.mark.parametrize("taps,flags", [("1", 0), ("n", CORR), ("n+3", CENTER)])
def test_rows(gpu, log2n, rows, taps, flags):
    n = 1 << log2n
    check(gpu, n, rows, {"1": 1, "n": n, "n+3": n + 3}[taps], flags)


@pytest.mark.parametrize("n,rows,k,flags", [
    (2 ** 14, 1, 1, 0),               # 2^13 windows: two a row, the second short
    (2 ** 14, 3, 4097, CORR),         # the longest filter of 2^13 windows
    (2 ** 14, 3, 33, CENTER),         # outputs wrap at the row's end
    (2 ** 14, 1, 4096, CENTER | CORR),
    (2 ** 15, 1, 8193, 0),            # 2^14 windows, the longest filter
    (2 ** 15, 3, 8193, CORR | CENTER),
    (2 ** 15, 1, 4098, CENTER),
    (2 ** 17, 5, 5000, CENTER),       # odd numbers of windows
])
def test_windows(gpu, n, rows, k, flags):
    check(gpu, n, rows, k, flags)
