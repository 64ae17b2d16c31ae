"""The built library's own gfx950 code, disassembled: what the compiler checks in the code it writes and cannot check in
instructions written by hand."""
import os
import re
import shutil
import struct
import subprocess
import tempfile

import pytest

from nextsycl_amd import library_path

LLVM = os.path.join(os.path.dirname(os.path.realpath(shutil.which("hipcc") or "/opt/rocm/bin/hipcc")), "..", "llvm", "bin")
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    """The gfx950 code objects of a host library: each bundle is a count and (offset, size, length of name, name) entries."""
    at = data.find(BUNDLE)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + len(BUNDLE))
        p = at + len(BUNDLE) + 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + n] and size:
                yield data[at + off:at + off + size]
            p += 24 + n
        at = data.find(BUNDLE, at + len(BUNDLE))


def _over_code_objects(tool, *args):
    """An LLVM tool's output over each code object of the library."""
    if not os.path.exists(library_path()):
        from nextsycl_amd.build import build
        build()
    out = []
    for obj in _code_objects(open(library_path(), "rb").read()):
        with tempfile.NamedTemporaryFile() as f:
            f.write(obj)
            f.flush()
            out.append(subprocess.run([os.path.join(LLVM, tool)] + list(args) + [f.name], capture_output=True, text=True, check=True).stdout)
    assert out
    return out


@pytest.fixture(scope="module")
def listing():
    """{kernel: [(opcode, operands)]} in program order."""
    kernels = {}
    for text in _over_code_objects("llvm-objdump", "-d", "--no-show-raw-insn"):
        code = None
        for line in text.split("\n"):
            head = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            if head:
                code = kernels.setdefault(head[1], [])
                continue
            ins = line.split("//")[0].split(None, 1)
            if code is not None and ins:
                code.append((ins[0], ins[1].strip() if len(ins) > 1 else ""))
    return kernels


def test_transfers_into_lds_wait_for_m0(listing):
    """A transfer from memory into LDS takes its LDS address from M0, and M0 written by the scalar unit takes one wait state
    to arrive: no transfer follows such a write directly."""
    found, bad = 0, {}
    for name, code in listing.items():
        for (op, args), (op2, args2) in zip(code, code[1:]):
            if "_load_lds_" in op2 or re.search(r"\blds\b", args2):
                found += 1
                if op.startswith("s_") and re.match(r"m0\b", args):
                    bad[name] = bad.get(name, 0) + 1
    assert found > 100 and not bad, bad
