"""The gfx950 code objects of libhpsp.so, read on the CPU: registers of every
kernel (from the metadata note) and its instructions (llvm-objdump)."""
import functools
import os
import struct
import subprocess
import tempfile

import msgpack

from hydra_amd import capi

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"
NT_AMDGPU_METADATA = 32


def elfs():
    data = open(capi.LIB_PATH, "rb").read()
    out, at = [], data.find(BUNDLE)
    while at >= 0:
        p = at + len(BUNDLE)
        (entries,) = struct.unpack_from("<Q", data, p)
        p += 8
        for _ in range(entries):
            off, size, name_len = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + name_len].decode()
            p += 24 + name_len
            if "gfx950" in name and size:
                out.append(data[at + off:at + off + size])
        at = data.find(BUNDLE, at + 1)
    return out


def metadata(elf):
    """The kernels' entries of the NT_AMDGPU_METADATA note."""
    (phoff,) = struct.unpack_from("<Q", elf, 32)
    size, count = struct.unpack_from("<HH", elf, 54)
    for i in range(count):
        h = struct.unpack_from("<IIQQQQQQ", elf, phoff + i * size)
        p, end = h[2], h[2] + h[5]
        while h[0] == 4 and p < end:  # PT_NOTE
            n, d, kind = struct.unpack_from("<III", elf, p)
            desc = p + 12 + (n + 3) // 4 * 4
            if kind == NT_AMDGPU_METADATA:
                return msgpack.unpackb(elf[desc:desc + d])["amdhsa.kernels"]
            p = desc + (d + 3) // 4 * 4
    return []


@functools.lru_cache(maxsize=None)
def kernels():
    """Mangled name -> (metadata, ELF image)."""
    return {k[".name"]: (k, e) for e in elfs() for k in metadata(e)}


def find(prefix):
    """The kernels whose mangled name starts with _ZN4hpsp<length><prefix>."""
    base = prefix.split("I")[0]
    head = f"_ZN4hpsp{len(base)}{prefix}"
    hits = {n: k for n, (k, _) in kernels().items() if n.startswith(head)}
    assert hits, head
    return hits


def waves(k):
    """Waves per SIMD that a kernel's vector registers allow (512 per lane)."""
    return min(8, 512 // ((k[".vgpr_count"] + 7) // 8 * 8))


def instructions(name):
    with tempfile.NamedTemporaryFile(suffix=".elf") as f:
        f.write(kernels()[name][1])
        f.flush()
        text = subprocess.run([OBJDUMP, "-d", f"--disassemble-symbols={name}", f.name], check=True,
                              capture_output=True, text=True).stdout
    return [line.split("//")[0].strip() for line in text.splitlines() if line.startswith("\t")]


def have_objdump():
    return os.path.exists(OBJDUMP)
