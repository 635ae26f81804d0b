"""What the compiler made of the built kernels, from the metadata in the library: the projections and what adds their slices up keep everything in registers.  A register that
goes to memory inside a weight stream costs a wait for all that is in flight, and kernels that carry code for other calls are how it happens."""
import struct

import msgpack
import pytest

from vllm_neuron_amd import _native


def kernels():
    """Name -> metadata of every kernel in the library's code objects (ELF files for machine 224, their notes of type 32)."""
    _native.load_library()
    with open(_native.LIB_PATH, "rb") as f:
        data = f.read()
    found, at = {}, data.find(b"\x7fELF", 1)
    while at >= 0:
        if struct.unpack_from("<H", data, at + 18)[0] == 224:
            table, (entry, count) = struct.unpack_from("<Q", data, at + 40)[0], struct.unpack_from("<HH", data, at + 58)
            for head in range(at + table, at + table + entry * count, entry):
                if struct.unpack_from("<I", data, head + 4)[0] != 7:      # notes
                    continue
                p, size = struct.unpack_from("<QQ", data, head + 24)
                p, end = p + at, p + at + size
                while p < end:
                    name, desc, kind = struct.unpack_from("<III", data, p)
                    p += 12 + (name + 3 & ~3)
                    if kind == 32:
                        found.update((k[".name"], k) for k in msgpack.unpackb(data[p:p + desc])["amdhsa.kernels"])
                    p += desc + 3 & ~3
        at = data.find(b"\x7fELF", at + 4)
    return found


@pytest.mark.parametrize("kernel", ["splitk_reduce_kernel", "gemm_wide", "gemv_", "attn_window_decode_kernel", "attn_decode_kernel"])
def test_nothing_in_scratch(kernel):
    mine = {n: k for n, k in kernels().items() if kernel in n}
    assert mine
    assert not [n for n, k in mine.items() if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]]
