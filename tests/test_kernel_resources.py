"""What the built library's kernels ask for, from their descriptors in its code objects (no GPU needed)."""
import os
import struct

import foundry_attn as fa

# Kept a few registers in memory since it was first measured, outside its loop.
KNOWN = {"panel_kernelILi8ELi2ELi1ELi2ELb1ELb0ELb0E": 12}


def _code_objects(data):
    at = data.find(b"__CLANG_OFFLOAD_BUNDLE__")
    while at >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", data, at + 24)[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + length]
            entry += 24 + length
            if b"gfx" in target and size:
                yield data[at + offset:at + offset + size]
        at = data.find(b"__CLANG_OFFLOAD_BUNDLE__", at + 24)


def _scratch(elf):
    """(kernel, bytes of memory per work-item that its registers do not hold), from the descriptor symbols NAME.kd."""
    table, = struct.unpack_from("<Q", elf, 0x28)
    entry, count = struct.unpack_from("<HH", elf, 0x3A)
    sections = [struct.unpack_from("<IIQQQQIIQQ", elf, table + i * entry) for i in range(count)]
    for s in sections:
        if s[1] != 11:  # the dynamic symbols
            continue
        names = sections[s[6]][4]
        for i in range(s[5] // 24):
            name, _, _, index, value, _ = struct.unpack_from("<IBBHQQ", elf, s[4] + 24 * i)
            text = elf[names + name:elf.index(b"\0", names + name)].decode()
            if text.endswith(".kd"):
                yield text[:-3], struct.unpack_from("<II", elf, sections[index][4] + value - sections[index][3])[1]


def test_no_kernel_keeps_registers_in_memory():
    with open(os.path.join(os.path.dirname(fa.__file__), "libfoundry_attn.so"), "rb") as f:
        kernels = [k for elf in _code_objects(f.read()) for k in _scratch(elf)]
    assert len(kernels) > 300  # (every instance of every template)
    assert {n: b for n, b in kernels if b and not any(k in n and b <= most for k, most in KNOWN.items())} == {}
