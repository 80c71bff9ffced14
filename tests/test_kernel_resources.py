"""What the compiled kernels hold, read from the metadata of the code objects in the library
(no GPU): no kernel keeps values in scratch memory.  A kernel with a few spilled registers
is not only slower for the spills: where a launch is short, so is the set-up of its scratch
(k_conv_ols with 24 bytes of it: 12.7 -> 14.5 us a call on a row of 2^14 values)."""
import os
import struct

import msgpack
import pytest

import estl_amd


def code_objects(blob):
    """The gfx950 ELF images embedded in the library (offload bundles, uncompressed)."""
    at = blob.find(b"\x7fELF", 4)
    while at >= 0:
        machine = struct.unpack_from("<H", blob, at + 18)[0]
        if machine == 224:  # EM_AMDGPU
            yield at
        at = blob.find(b"\x7fELF", at + 4)


def kernels(blob, base):
    """The kernel descriptors (msgpack, NT_AMDGPU_METADATA) of the image at `base`."""
    shoff, = struct.unpack_from("<Q", blob, base + 40)
    entsize, count = struct.unpack_from("<HH", blob, base + 58)
    for i in range(count):
        sh = base + shoff + i * entsize
        kind, = struct.unpack_from("<I", blob, sh + 4)
        off, size = struct.unpack_from("<QQ", blob, sh + 24)
        if kind != 7:  # SHT_NOTE
            continue
        p, end = base + off, base + off + size
        while p < end:
            namesz, descsz, ntype = struct.unpack_from("<III", blob, p)
            desc = p + 12 + (namesz + 3) // 4 * 4
            if ntype == 32:
                meta = msgpack.unpackb(blob[desc:desc + descsz], strict_map_key=False)
                yield from meta["amdhsa.kernels"]
            p = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def found():
    if not os.path.exists(estl_amd.LIB_PATH):
        pytest.skip("library not built")
    with open(estl_amd.LIB_PATH, "rb") as f:
        blob = f.read()
    all_kernels = [k for base in code_objects(blob) for k in kernels(blob, base)]
    assert len(all_kernels) > 100, "no kernel metadata found in the library"
    return all_kernels


def test_no_kernel_uses_scratch(found):
    spilled = {k[".name"]: k[".private_segment_fixed_size"] for k in found if k[".private_segment_fixed_size"]}
    assert not spilled, spilled


def test_work_queue_reads_arguments_where_needed(found):
    """The arguments of all size classes do not fit the scalar registers: read ahead of the work
    loop, they are spilled by the dozen, with a wait for each group of them (52 spilled, 0.7 us a
    call)."""
    counts = [k[".sgpr_spill_count"] for k in found if "k_ubatch" in k[".name"]]
    assert len(counts) == 2 and max(counts) <= 8, counts
