"""The device code of the built library: kernels' instructions and resources, by symbol."""
import os
import re
import struct
import subprocess
import tempfile

import pytest

from neuralangelo_amd import build

LLVM = "/opt/rocm/llvm/bin/"


def code_objects():
    """The gfx950 code objects in the library's offload bundles."""
    with tempfile.TemporaryDirectory() as tmp:
        fat = os.path.join(tmp, "fat")
        subprocess.run([LLVM + "llvm-objcopy", "--dump-section", f".hip_fatbin={fat}",
                        build.LIB_PATH, os.path.join(tmp, "copy")], check=True)
        with open(fat, "rb") as f:
            data = f.read()
    magic, at, out = b"__CLANG_OFFLOAD_BUNDLE__", 0, []
    while (at := data.find(magic, at)) >= 0:
        (count,) = struct.unpack_from("<Q", data, at + len(magic))
        o = at + len(magic) + 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, o)
            if build.ARCH.encode() in data[o + 24:o + 24 + n] and size:
                out.append(data[at + off:at + off + size])
            o += 24 + n
        at += len(magic)
    return out


def _run(tool, obj, *args):
    with tempfile.NamedTemporaryFile(suffix=".o") as f:
        f.write(obj)
        f.flush()
        return subprocess.run([LLVM + tool, *args, f.name], check=True, capture_output=True,
                              text=True).stdout


def kernels(pattern):
    """{symbol: [(address, mnemonic, operands, branch target or None)]} of matching kernels."""
    found = {}
    for obj in code_objects():
        if re.search(pattern, obj.decode("latin-1")) is None:
            continue
        code = None
        for line in _run("llvm-objdump", obj, "-d", "--no-show-raw-insn").splitlines():
            if m := re.match(r"([0-9a-f]+) <(\S+)>:", line):
                code, start = (found.setdefault(m[2], []) if re.search(pattern, m[2]) else None), int(m[1], 16)
            elif code is not None and (m := re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]+):(.*)", line)):
                to = re.search(r"<[^+>]+(?:\+0x([0-9a-f]+))?>", m[4]) if "branch" in m[1] else None
                code.append((int(m[3], 16), m[1], m[2], start + int(to[1] or "0", 16) if to else None))
    if not found:
        pytest.fail(f"no kernel matches {pattern}")
    return found


def resources(pattern):
    """{symbol: {field: number}} from the metadata of matching kernels."""
    found = {}
    for obj in code_objects():
        notes = _run("llvm-readelf", obj, "--notes")
        for block in re.split(r"\n  - (?=\.)", notes):
            name = re.search(r"\.name:\s+(_Z\S+)", block)
            if name and re.search(pattern, name[1]):
                found[name[1]] = {k: int(v) for k, v in re.findall(r"\.(\w+):\s+(\d+)\n", block)}
    if not found:
        pytest.fail(f"no kernel matches {pattern}")
    return found


def waits(operands):
    """(vmcnt, lgkmcnt) of an s_waitcnt; None where it does not wait for one."""
    def count(name):
        m = re.search(name + r"\((\d+)\)", operands)
        return int(m[1]) if m else None
    return count("vmcnt"), count("lgkmcnt")
