"""Infinite inputs of transforms that are one register DFT (2 to 16 values): every part of a bin
that the infinity reaches is infinite with the sign of its cosine or sine, no part is NaN, and
the parts that it does not reach hold the rest of the sum.  (Longer transforms hand infinities
through products with table values, and give NaN.)"""
import numpy as np
import pytest

import estl_amd

pytestmark = pytest.mark.gpu


def transform(gpu, x, direction):
    import torch
    d = torch.from_numpy(x).to(gpu)
    y = torch.empty_like(d)
    estl_amd.Plan(x.shape[1], x.shape[0], direction).execute(d, y)
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("n", [2, 4, 8, 16])
@pytest.mark.parametrize("direction", [estl_amd.FORWARD, estl_amd.BACKWARD])
@pytest.mark.parametrize("imag", [False, True])
def test_one_infinity(gpu, n, direction, imag):
    rng = np.random.default_rng(5)
    base = (rng.uniform(-1, 1, (n, n)) + 1j * rng.uniform(-1, 1, (n, n))).astype(np.complex64)
    x = base.copy()
    for j in range(n):  # row j: the infinity in value j
        part = x[j].view(np.float32)
        part[2 * j + imag] = np.inf
        base[j].view(np.float32)[2 * j + imag] = 0.0
    got = transform(gpu, x, direction)
    rest = base.astype(np.complex128) @ np.exp(direction * 2j * np.pi * np.outer(np.arange(n), np.arange(n)) / n)
    w = np.exp(direction * 2j * np.pi * np.outer(np.arange(n), np.arange(n)) / n) * (1j if imag else 1)
    for parts, weight, finite in ((got.real, w.real, rest.real), (got.imag, w.imag, rest.imag)):
        reached = np.abs(weight) > 1e-9
        assert np.array_equal(parts[reached], np.where(weight[reached] > 0, np.inf, -np.inf).astype(np.float32))
        assert np.allclose(parts[~reached], finite[~reached], rtol=0, atol=1e-6 * n)
