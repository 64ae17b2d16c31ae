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


def _vector_registers(operand):
    m = re.match(r"[-|]*([va])(?:\[(\d+):(\d+)\]|(\d+))", operand.strip())
    return {(m[1], i) for i in range(int(m[2] or m[4]), int(m[3] or m[4]) + 1)} if m else set()


def test_matrix_results_are_met_by_their_wait_states(listing):
    """A 16 x 16 x 32 matrix instruction of 16-bit operands takes four passes: for 8 wait states a vector instruction may neither
    read nor write its result, for 3 it may not write the registers of its third operand. The compiler keeps these between
    instructions of its own and cannot keep them for a vector instruction written by hand. (Along straight lines of code; a
    matrix instruction's own rules are others.)"""
    found, bad = 0, {}
    for name, code in listing.items():
        clock, live = 0, []                                   # live: (state behind it, its result, its third operand's registers)
        for op, args in code:
            if op == "s_nop":
                clock += int(args, 0) + 1
                continue
            if op in ("s_branch", "s_endpgm", "s_setpc_b64"):
                live = []
            live = [x for x in live if clock - x[0] < 8]
            operands = re.split(r",\s*(?![^\[]*\])", args)
            if op.startswith("v_mfma"):
                if "16x16x32" in op:
                    found += 1
                    live.append((clock + 1, _vector_registers(operands[0]), _vector_registers(operands[3])))
            elif live and op.startswith("v_"):
                scalar = op.startswith(("v_cmp", "v_readfirstlane", "v_readlane"))
                write = set() if scalar else _vector_registers(operands[0])
                touched = set().union(write, *[_vector_registers(x) for x in operands])
                for at, result, third in live:
                    if touched & result or (clock - at < 3 and write & third):
                        bad.setdefault(name, []).append("%s %s" % (op, args))
            clock += 1
    assert found > 1000 and not bad, bad


@pytest.fixture(scope="module")
def spilled():
    """{kernel: vector registers spilled}"""
    out = {}
    for text in _over_code_objects("llvm-readelf", "--notes"):
        for kernel in text.split("\n  - .agpr_count:")[1:]:
            out[re.search(r"^    \.name: +(\S+)$", kernel, re.M)[1]] = int(re.search(r"\.vgpr_spill_count: +(\d+)", kernel)[1])
    return out


def test_decode_over_quantized_rows_of_256_spills_nothing(spilled):
    """Its counted waits leave transfers in flight over a tile's arithmetic; a register's way back from memory would wait for
    all of them."""
    form = {name: n for name, n in spilled.items() if "attn_decode_q256_kernel" in name}
    assert len(form) == 4 and not any(form.values()), form


def test_two_row_tiles_over_bfloat16_rows_of_256_spill_no_more(spilled):
    """The merge of two row tiles as they lie takes no registers over the tile loop: 36 are spilled there in row order, 44 where its places are kept."""
    form = [n for name, n in spilled.items() if "attn_decode_kernelILi256ELi2ELi3ELb0E" in name]
    assert len(form) == 1 and form[0] <= 37, form


def test_prompt_kernels_spill_no_vector_registers_over_a_tile(spilled):
    """Their counted waits leave transfers in flight over a tile's arithmetic too. Rows in two parts laid end to end spill a row's place, written
    before the tiles and read behind the last: 2 registers at heads of 128, 5 at 256; no other instance spills any."""
    form = {name: n for name, n in spilled.items() if "attn_prefill" in name}
    two = {name: n for name, n in form.items() if re.search(r"attn_prefill_flat_kernelILi(128|256)ELb1ELi0ELb1E", name)}
    assert len(form) > 20 and len(two) == 2 and all(n <= (2 if "ILi128E" in name else 5) for name, n in two.items()), two
    assert not any(n for name, n in form.items() if name not in two), {name: n for name, n in form.items() if n}
