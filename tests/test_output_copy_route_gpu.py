"""Which copies of a served output the streaming copy's kernel takes (launch_output_copy, called
directly): 8 MiB and more, whole 16-byte values on 16-byte boundaries, inside one
allocation of the device; the rest it leaves to the runtime, with no error recorded that a
later launch would report."""
import ctypes

import pytest

import estl_amd

pytestmark = pytest.mark.gpu

MIN = 8 << 20


def test_output_copy_route(gpu):
    import torch
    f = getattr(estl_amd.lib(), "_ZN4estl18launch_output_copyEPKvPvmiP12ihipStream_tPb")
    f.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_void_p,
                  ctypes.POINTER(ctypes.c_bool)]
    f.restype = ctypes.c_int
    last = estl_amd.lib().hipGetLastError  # of the runtime the library is linked to

    def route(src, dst, size, stream=None):
        queued = ctypes.c_bool(True)
        assert f(src, dst, size, 0, stream, ctypes.byref(queued)) == 0
        assert last() == 0
        return queued.value

    n = MIN + 4096
    src = torch.randint(0, 256, (n,), dtype=torch.uint8, device=gpu)
    dst = torch.zeros(n, dtype=torch.uint8, device=gpu)
    host = torch.zeros(n, dtype=torch.uint8)
    pinned = torch.zeros(n, dtype=torch.uint8, pin_memory=True)
    torch.cuda.synchronize()
    s, d = src.data_ptr(), dst.data_ptr()
    for stream in (None, torch.cuda.Stream().cuda_stream):
        dst.zero_()
        torch.cuda.synchronize()
        assert route(s, d + 16, MIN, stream)
        torch.cuda.synchronize()
        assert torch.equal(dst[16:16 + MIN], src[:MIN]) and not dst[:16].any() and not dst[16 + MIN:].any()
    assert not route(s, d, MIN - 16)
    assert not route(s, d, MIN + 8)
    assert not route(s, d + 8, MIN)
    assert not route(s + 8, d, MIN)
    assert not route(s, host.data_ptr() + (-host.data_ptr()) % 16, MIN)
    assert not route(s, pinned.data_ptr(), MIN)
    assert not route(s, d, 1 << 40)  # past the allocation: left to the runtime, which refuses it
    torch.cuda.synchronize()
