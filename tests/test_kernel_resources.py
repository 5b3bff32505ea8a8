"""What the built kernels take of a compute unit, from the metadata of the code object inside the library: kernels that keep their
operands in registers must not send them through scratch memory."""
import os
import re
import struct

import msgpack
import pytest


def _kernels():
    """Metadata of every kernel by mangled name: the offload bundles of the library hold ELF files, whose note of type 32 is a msgpack map."""
    from m2_amd import _lib
    with open(_lib.LIB_PATH, "rb") as f:
        data = f.read()
    found = {}
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at, (count,) = m.start() + 32, struct.unpack_from("<Q", data, m.start() + 24)
        for _ in range(count):
            off, size, name = struct.unpack_from("<QQQ", data, at)
            triple, at = data[at + 24:at + 24 + name], at + 24 + name
            elf = data[m.start() + off:m.start() + off + size]
            if b"gfx950" not in triple:
                continue
            headers, (each, number) = struct.unpack_from("<Q", elf, 0x28)[0], struct.unpack_from("<HH", elf, 0x3A)
            for i in range(number):
                kind, (start, length) = struct.unpack_from("<I", elf, headers + i * each + 4)[0], struct.unpack_from("<QQ", elf, headers + i * each + 24)
                note = start
                while kind == 7 and note < start + length:
                    name_size, desc_size, note_type = struct.unpack_from("<III", elf, note)
                    note += 12 + (name_size + 3) // 4 * 4
                    if note_type == 32:
                        for k in msgpack.unpackb(elf[note:note + desc_size], strict_map_key=False)["amdhsa.kernels"]:
                            found[k[".name"]] = k
                    note += (desc_size + 3) // 4 * 4
    return found


@pytest.mark.parametrize("kernel", ["project_kernel", "hidden_kernel", "project_spectrum_kernel", "mixer_pair_kernel", "mixer_long_kernel", "conv_real_kernel",
                                    "small_gemm_kernel", "ln_gemm_kernel", "layernorm_kernel", "pooler_kernel"])
def test_kernels_without_scratch(kernel):
    mine = {n: k for n, k in _kernels().items() if f"{len(kernel)}{kernel}" in n}
    assert mine, kernel
    assert not {n: k[".private_segment_fixed_size"] for n, k in mine.items() if k[".private_segment_fixed_size"]}


def test_scratch_of_the_longest_rows():
    """mixer_real_kernel holds a row in up to 192 of its 256 registers; a few loads of spilled factors a row are what it may take."""
    mine = {n: k[".private_segment_fixed_size"] for n, k in _kernels().items() if "17mixer_real_kernel" in n}
    assert len(mine) == 4 and max(mine.values()) <= 16, mine
