"""What the compiler gave kernels whose launches count on it: registers and spills, read from the kernel descriptions that
the built library carries (no GPU)."""

import re
import struct

import msgpack
import pytest

from tensorfold_amd import build


@pytest.fixture(scope="module")
def kernels():
    """{mangled name: description} over the gfx950 code objects of libtfmi.so."""

    build.load()
    blob, found = build.LIB.read_bytes(), {}
    for bundle in re.finditer(rb"__CLANG_OFFLOAD_BUNDLE__", blob):
        at = bundle.start()
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", blob, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", blob, entry)
            target = blob[entry + 24:entry + 24 + length]
            entry += 24 + length
            if not target.endswith(build.ARCH.encode()):
                continue
            elf = blob[at + offset:at + offset + size]
            table, = struct.unpack_from("<Q", elf, 40)
            each, count = struct.unpack_from("<HH", elf, 58)
            for section in range(table, table + each * count, each):
                if struct.unpack_from("<I", elf, section + 4)[0] != 7:            # SHT_NOTE
                    continue
                note, = struct.unpack_from("<Q", elf, section + 24)
                name_size, size, kind = struct.unpack_from("<III", elf, note)
                if kind == 32:                                                     # NT_AMDGPU_METADATA
                    start = note + 12 + (name_size + 3) // 4 * 4
                    found.update({k[".name"]: k for k in msgpack.unpackb(elf[start:start + size])["amdhsa.kernels"]})
    assert found
    return found


def arguments(kernels, name):
    """[(integer template arguments, description)] of the instances of a kernel."""

    mangled = re.compile(rf"{len(name)}{name}I((?:L[a-z]\d+E)+)E")
    hits = [(tuple(map(int, re.findall(r"L[a-z](\d+)E", m[1]))), k) for n, k in kernels.items() if (m := mangled.search(n))]
    assert hits
    return hits


def test_two_workgroups_of_eight_waves_of_an_exl3_layer_share_a_compute_unit(kernels):
    """Four waves a SIMD (128 of its 512 registers each, accumulators among them) at every width, without spills."""

    seen = arguments(kernels, "linear_kernel")
    assert {a[0] for a, _ in seen} == {2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16}
    over = {a: (k[".vgpr_count"], k[".vgpr_spill_count"]) for a, k in seen if k[".vgpr_count"] > 128 or k[".vgpr_spill_count"]}
    assert not over
