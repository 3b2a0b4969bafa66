"""What the compiler recorded of each kernel in a library built from this repository's
sources: registers, scratch and LDS from the code objects' metadata notes."""
import struct
import subprocess

import msgpack

NT_AMDGPU_METADATA = 32


def _elves(data):
    """The gfx950 code objects of every offload bundle in the file."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(magic)
    while at >= 0:
        pos = at + len(magic)
        (n,) = struct.unpack_from("<Q", data, pos)
        pos += 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, pos)
            pos += 24
            ident = data[pos:pos + idlen]
            pos += idlen
            if b"gfx950" in ident:
                yield data[at + off:at + off + size]
        at = data.find(magic, at + 1)


def _notes(elf):
    phoff, = struct.unpack_from("<Q", elf, 32)
    phentsize, phnum = struct.unpack_from("<HH", elf, 54)
    for k in range(phnum):
        kind, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + k * phentsize)
        if kind != 4:  # PT_NOTE
            continue
        end = off + size
        while off < end:
            nlen, dlen, t = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (nlen + 3) // 4 * 4
            yield t, elf[desc:desc + dlen]
            off = desc + (dlen + 3) // 4 * 4


def kernels(path):
    """{demangled kernel name without arguments: metadata dict}"""
    with open(path, "rb") as f:
        data = f.read()
    found = []
    for elf in _elves(data):
        for t, desc in _notes(elf):
            if t == NT_AMDGPU_METADATA:
                found += msgpack.unpackb(desc)["amdhsa.kernels"]
    names = subprocess.run(["c++filt"], input="\n".join(k[".name"] for k in found),
                           capture_output=True, text=True, check=True).stdout.splitlines()
    clean = (n[:n.rindex("(")].replace("void ", "").replace("va::", "").strip()
             if "(" in n else n for n in names)
    return dict(zip(clean, found))
