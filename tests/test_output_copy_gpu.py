"""A served request's output copied out whole, in parts and to any address: the copy's
kernel takes 8 MiB and more of 16-byte values on 16-byte boundaries of one device, the
runtime the rest.
Bytes, so the comparison is exact."""
import pytest

import estl_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rows", [(2, 1), (1 << 10, 2047), (1 << 10, 2048), (1 << 14, 129), (1 << 20, 9)])
def test_output_copy(gpu, n, rows):
    import torch
    x = torch.empty(rows, n, dtype=torch.float32, device=gpu)
    h = torch.empty(min(n, 17), dtype=torch.float32, device=gpu)
    estl_amd.fill_uniform(x, 1)
    estl_amd.fill_uniform(h, 2)
    srv = estl_amd.Server(1 << 28, streams=2)
    try:
        rid = srv.submit_conv(n, rows, x, h)
        srv.wait(rid)
        size = 4 * n * rows
        side = torch.cuda.Stream()
        conv = estl_amd.Convolution(n, rows)
        conv.set_filter(h)
        y = torch.empty_like(x)
        conv.execute(x, y)
        torch.cuda.synchronize()
        want = y.view(-1).view(torch.uint8)
        for shift in (0, 4, 16):
            for count in {size, size - 4, size - 1, 16, 1}:
                if not 0 < count <= size:
                    continue
                for stream in (None, side):
                    dst = torch.full((size + 64,), 0xA5, dtype=torch.uint8, device=gpu)
                    torch.cuda.synchronize()
                    estl_amd.check(estl_amd.lib().estl_server_copy_output(
                        srv._h, rid, dst.data_ptr() + shift, count, estl_amd._stream_ptr(stream)))
                    torch.cuda.synchronize()
                    assert torch.equal(dst[shift:shift + count], want[:count]), (shift, count)
                    assert bool((dst[:shift] == 0xA5).all()) and bool((dst[shift + count:] == 0xA5).all())
        with pytest.raises(estl_amd.EstlError):  # more than the output's block holds
            estl_amd.check(estl_amd.lib().estl_server_copy_output(
                srv._h, rid, dst.data_ptr(), size + (1 << 20), estl_amd._stream_ptr(None)))
        srv.release(rid)
    finally:
        srv.close()
