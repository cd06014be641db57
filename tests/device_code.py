"""The gfx950 code objects inside a built shared library (helpers of the tests
that check the compiler's output)."""
import os
import re
import struct
import subprocess

LLVM = "/opt/rocm/llvm/bin"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 ELF images of every offload bundle in the library."""
    data = open(path, "rb").read()
    out, at = [], data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        pos = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + idlen].decode()
            pos += 24 + idlen
            if "gfx950" in name and size:
                out.append(data[at + off:at + off + size])
        at = data.find(MAGIC, at + 1)
    return out


def kernel_metadata(path, tmp_path):
    """{kernel name (mangled): {key: int}} of the integer entries of each
    kernel's metadata."""
    kernels = {}
    for i, img in enumerate(code_objects(path)):
        f = tmp_path / f"{i}.co"
        f.write_bytes(img)
        text = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", str(f)],
                              capture_output=True, text=True, check=True).stdout
        for block in re.split(r"\n  - \.agpr_count", text)[1:]:
            name = re.search(r"\.name:\s+(\S+)", block).group(1)
            kernels[name] = {k: int(v) for k, v in
                             re.findall(r"\.(\w+):\s+(\d+)\s*$", block, re.M)}
    return kernels


def disassemble(path, tmp_path, pattern):
    """(symbol, [instruction text]) of the kernels whose mangled name matches."""
    for i, img in enumerate(code_objects(path)):
        f = tmp_path / f"{i}.co"
        f.write_bytes(img)
        syms = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "-sW", str(f)],
                              capture_output=True, text=True, check=True).stdout
        names = sorted({s.split()[-1] for s in syms.splitlines()
                        if " FUNC " in s and re.search(pattern, s.split()[-1])})
        if not names:
            continue
        text = subprocess.run([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn",
                               "--no-leading-addr", "--disassemble-symbols=" + ",".join(names),
                               str(f)], capture_output=True, text=True, check=True).stdout
        for block in re.split(r"\n(?=(?:[0-9a-f]+ )?<\S+>:)", text):
            m = re.match(r"(?:[0-9a-f]+ )?<(\S+)>:", block)
            if m:
                yield m.group(1), [ln.split("//")[0].strip() for ln in
                                   block.splitlines()[1:] if ln.strip()]
