"""Registers and scratch memory of the compiled kernels whose launch rules
count on them: the compiler's metadata in the built library (no GPU needed)."""
import os
import struct

import msgpack
import pytest

from conftest import ROOT


def kernels():
    """{mangled name: metadata} of every gfx950 kernel in libkk.so."""
    path = os.path.join(ROOT, "best-tts-godot_amd", "libkk.so")
    if not os.path.exists(path):
        pytest.skip("libkk.so is not built")
    data = open(path, "rb").read()
    found, at = {}, 0
    while (at := data.find(b"\x7fELF\x02\x01", at + 1)) > 0:
        if struct.unpack_from("<H", data, at + 18)[0] != 224:  # EM_AMDGPU
            continue
        shoff, = struct.unpack_from("<Q", data, at + 40)
        shsize, shnum = struct.unpack_from("<HH", data, at + 58)
        for i in range(shnum):
            kind, off = struct.unpack_from("<4xI16xQ", data, at + shoff + i * shsize)
            if kind != 7:  # SHT_NOTE
                continue
            namesz, descsz, note = struct.unpack_from("<III", data, at + off)
            if note == 32:  # NT_AMDGPU_METADATA
                d = at + off + 12 + (namesz + 3) // 4 * 4
                for k in msgpack.unpackb(data[d:d + descsz])["amdhsa.kernels"]:
                    found[k[".name"]] = k
    return found


@pytest.mark.parametrize("name,vgprs", [
    # four blocks of four waves a CU share the launches of two to four a CU
    ("conv_i8_kernelILi2ELi2ELi1ELi1ELi3E", 128),
    # three
    ("conv_i8_kernelILi2ELi2ELi1ELi2ELi3E", 168),
    # eight waves a SIMD: short axes live on them
    ("reduce_generic_kernel", 64)])
def test_registers(name, vgprs):
    mine = {n: k for n, k in kernels().items() if name in n}
    assert mine, f"no kernel {name}"
    for n, k in mine.items():
        assert k[".vgpr_count"] <= vgprs, f"{n}: {k['.vgpr_count']} registers"
        assert k[".private_segment_fixed_size"] == 0, f"{n}: scratch memory"
