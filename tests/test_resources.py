"""What the compiler gave the kernels of the built library, read from the
metadata of its device image: no kernel that the granularity rule can pick
keeps registers in scratch memory."""
import struct

import msgpack

import xted

NOTE = 7  # ELF section type


def kernel_metadata(path):
    """{kernel name: its metadata} over the device images bundled in a library."""
    data = open(path, "rb").read()
    out, pos = {}, data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while pos >= 0:
        count, = struct.unpack_from("<Q", data, pos + 24)
        at = pos + 32
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx" not in target or not size:
                continue
            image = data[pos + offset:pos + offset + size]
            sections, = struct.unpack_from("<Q", image, 40)
            entry, number = struct.unpack_from("<HH", image, 58)
            for i in range(number):
                head = sections + i * entry
                if struct.unpack_from("<I", image, head + 4)[0] != NOTE:
                    continue
                note, = struct.unpack_from("<Q", image, head + 24)
                name_len, desc_len = struct.unpack_from("<II", image, note)
                desc = note + 12 + (name_len + 3 & ~3)
                meta = msgpack.unpackb(image[desc:desc + desc_len], strict_map_key=False)
                out.update({k[".name"]: k for k in meta["amdhsa.kernels"]})
        pos = data.find(b"__CLANG_OFFLOAD_BUNDLE__", pos + 24)
    return out


def test_no_form_the_rule_picks_spills():
    kernels = kernel_metadata(xted.LIB_PATH)
    assert sum("scan_kernel" in name for name in kernels) >= 50
    # 16 waves of 16 columns per lane are only ever forced (class 25).
    spilled = {name: k[".private_segment_fixed_size"] for name, k in kernels.items()
               if k[".private_segment_fixed_size"] and "scan_kernelILi16ELi16E" not in name}
    assert not spilled
