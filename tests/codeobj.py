"""The gfx950 code objects inside the library built from csrc/: kernel names with the registers, scratch and LDS the
compiler gave them, and a kernel's instructions."""
import os
import re
import struct
import subprocess
import tempfile

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen27-engine_amd", "lib", "libq27h.so")
LLVM = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _tool(name, *args):
    path = os.path.join(LLVM, name)
    if not os.path.exists(path):
        pytest.skip(f"{path} is not installed")
    return subprocess.run([path, *args], check=True, capture_output=True, text=True).stdout


def code_objects(lib=LIB):
    """The gfx950 ELF images of the library, one per translation unit with kernels."""
    with open(lib, "rb") as f:
        b = f.read()
    out, i = [], b.find(MAGIC)
    while i >= 0:
        n, = struct.unpack_from("<Q", b, i + len(MAGIC))
        p = i + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", b, p)
            if b"gfx950" in b[p + 24: p + 24 + idlen]:
                out.append(b[i + off: i + off + size])
            p += 24 + idlen
        i = b.find(MAGIC, i + 1)
    assert out, f"no gfx950 code object in {lib}"
    return out


def kernels(lib=LIB):
    """{mangled name: {"vgpr_count", "vgpr_spill_count", "private_segment_fixed_size", "group_segment_fixed_size"}}."""
    out = {}
    for image in code_objects(lib):
        with tempfile.NamedTemporaryFile(suffix=".co") as f:
            f.write(image)
            f.flush()
            notes = _tool("llvm-readelf", "--notes", f.name)
        for k in notes.split("- .agpr_count:")[1:]:
            out[re.search(r"\.name:\s+(\S+)", k).group(1)] = {
                x: int(re.search(rf"\.{x}:\s+(\d+)", k).group(1))
                for x in ("vgpr_count", "vgpr_spill_count", "private_segment_fixed_size", "group_segment_fixed_size")}
    return out


def instructions(kernel, lib=LIB):
    """The instructions of the one kernel whose mangled name contains `kernel`."""
    for image in code_objects(lib):
        if kernel.encode() not in image:
            continue
        with tempfile.NamedTemporaryFile(suffix=".co") as f:
            f.write(image)
            f.flush()
            text = _tool("llvm-objdump", "-d", "--no-show-raw-insn", f.name)
        for body in re.split(r"\n(?=[0-9a-f]+ <)", text):
            head, _, rest = body.partition("\n")
            if kernel in head:
                return [ln.split("//")[0].strip() for ln in rest.splitlines() if ln.strip()]
    raise AssertionError(f"kernel {kernel} is not in {lib}")
